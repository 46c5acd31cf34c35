// Subgraph traversal for gfx950: graph preparation and the per-query search.
//
// One wavefront (64 lanes, one workgroup) runs one query and reproduces, step
// for step, what the reference's host search does for that query
// (extension/traverse_cpu.cpp:12-163):
//   * the open list is the same array heap, with the same sift rules
//     (extension/inc/heapq.cuh:13-88): its top nine levels sit in registers,
//     where a pop or an insert changes a whole path at once, the rest in LDS
//     (search_lists.h);
//   * the result list is the exact set of the H best distances seen so far —
//     what the reference's result heap holds — as sorted keys in registers
//     (ResultKeys) and a log of the admitted candidates in device memory, from
//     which the set's nodes are read back at the end (ResultLog);
//   * the visited set is exact: one bit per storage row, in LDS where the
//     queries of a launch all run at once with so much of it (NEAR), else in a
//     per-wavefront slice of a pooled HBM bitmask (atomic OR), behind a small
//     LDS table of rows already known to be marked;
//   * a distance is the reference's eight-accumulator FMA sum
//     (extension/inc/distance.h:31-55) bit for bit: four lanes share a row,
//     lane a of the quad owns accumulators 2a and 2a+1 and streams its 16
//     bytes of every 64-byte block of the row (rows are in the layout of
//     pa_rows_prepare: the pairs of two groups of eight interleaved by lane).
// Expansion of a node therefore costs one coalesced row of neighbour ids, an
// atomic for each neighbour the LDS table does not know and one coalesced
// 4*dp-byte row per unvisited neighbour, 16 rows in flight per pass (32 where
// rows are 128 floats long).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <map>
#include <mutex>
#include <tuple>

#include "device_common.h"
#include "pilotann.h"
#include "search_lists.h"

using namespace pa;

namespace {

// ---- the search ---------------------------------------------------------------

struct TraverseArgs {
    int64_t *out_I;
    float *out_D;
    const int32_t *adj;
    const int32_t *gid;
    const int64_t *mapping;
    const float *storage;
    const float *query;
    const int64_t *init_I;
    const float *init_D;
    uint32_t *seen;
    int *work_counter;
    unsigned long long *counters;
    int batch, n_nodes, n_storage, dp, n_init, k, H, deg, max_iter;
    int words_per_slot, slot_stride, sort_n;
};

__global__ void reset_work_counter(int *counter) { *counter = 0; }

// Optional per-phase cycle tally for tuning builds (-DPA_PHASE_TIMERS): adds
// seven words after the five work counters.
#ifdef PA_PHASE_TIMERS
#define PA_TIMER_BEGIN() unsigned long long t_mark_ = __builtin_readcyclecounter()
#define PA_TIMER(i)                                                  \
    do {                                                             \
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); \
        unsigned long long t_now_ = __builtin_readcyclecounter();    \
        phase[i] += t_now_ - t_mark_;                                \
        t_mark_ = t_now_;                                            \
    } while (0)
#else
#define PA_TIMER_BEGIN() do {} while (0)
#define PA_TIMER(i) do {} while (0)
#endif

// Wavefronts per SIMD the register allocator must fit.  A budget a few
// registers under what the code needs costs more (spills, serialised loads)
// than the extra wavefront brings, so only a floor is given, under which no
// instance has to be squeezed (the largest heaps are bounded by their LDS
// anyway), and the allocator's own count decides the residency above it: 8 for
// the smallest instances, 3 for 128-float rows with two passes of loads in flight
// (TWO), which take 64 registers.  Measured for those on 250 000 rows of a million, four
// wavefronts (128 registers) / three (155 - 168), ms: H = 128, 1500 queries 0.72 / 0.64, 3000
// 1.01 / 0.93, 10 000 2.88 / 2.61; H = 256, 1500 1.58 / 1.11, 10 000 5.79 / 4.66.  With one pass,
// which is for launches that fill the device, five (96, up to 17 spilled) against
// four (103 - 115): 500 000 rows, H = 256, 10 000 queries 3.22 -> 3.10 ms, the other
// sizes within 1 % (64-float rows at H = 256, 103 registers: four 2.24, five 2.27
// ms, so no floor there).  H = 512 and 1024 with two passes need 172 - 183 and are
// held to three wavefronts (168, up to 17 spilled), which LDS then allows.
// Rows of a length without a kernel of its own need 133 - 137 at H = 384 and 512 and
// 175 at H = 2048: held to four wavefronts and to three (up to 8 spilled), without
// which, 75 000 rows of 40 floats, 10 000 queries, H = 384 took 3.73 ms, now 3.23; 512
// 5.20 / 4.48; 2048 28.0 / 25.3; 300 000 rows of 96 floats 5.01 / 4.66, 7.12 / 6.65, 36.2 / 34.0.
#ifdef PA_WAVES_PER_EU
#define PA_OCCUPANCY(H, WAVES) __attribute__((amdgpu_waves_per_eu(PA_WAVES_PER_EU, PA_WAVES_PER_EU)))
#else
#define PA_OCCUPANCY(H, WAVES) __attribute__((amdgpu_waves_per_eu((WAVES) > 1 && (H) <= 512 ? 4 : (H) <= 256 ? (TWO ? 3 : DP8 == 16 ? 5 : 4) : (H) <= 512 ? (DP8 == 0 ? 4 : 3) : (H) <= 1024 ? (TWO ? 3 : 2) : DP8 == 0 ? 3 : 1, 8)))
#endif

// The longest open list (4096 cells) keeps level 11 in the wavefront's region of
// device memory instead of LDS (search_lists.h): first level kept there, 0 = the
// whole list in registers and LDS.  Measured on 250 000 rows of 128 floats, 10 000
// queries: lists of 4096 cells run in 22.2 ms so (10 wavefronts a compute unit, one pass of
// rows), in 26.0 with all of it in LDS (5) and in 24.0 with level 10 there too; 3000
// queries 8.9, 9.1 and 7.4.  (Where all have room with the list in LDS, it is the faster:
// 1000 queries 4.33 / 3.32.)  Lists of 2048 cells: 8.9 ms in LDS, 11.0 with level 10 in
// device memory.
constexpr int deep_from(int H) { return H == 2048 ? 11 : 0; }

// NEAR: the visited bits of a query are in LDS (behind the query where that is
// dynamic too), without a table in front of them: for launches whose queries
// all run at once with so much LDS each (make_plan).  TWO: two passes of rows are
// read at a time.
//
// WAVES > 1 (with NEAR): the wavefront of a query has WAVES - 1 helpers, which read
// the neighbour ids and the rows of nodes it is about to expand and hand it the
// distances (LookAhead).  What is left to it, and bounds it, is the list work:
// 128-float rows, H = 128, one query, cycles an expansion 4600 -> 2900, of which the
// 2.6 inserts 1130, the pop 310.  It needs no registers for rows: 116 in place of 153,
// four wavefronts a SIMD.
template <int H, int DP8, bool NEAR, bool TWO, int WAVES>
__global__ __launch_bounds__(kWave *WAVES) PA_OCCUPANCY(H, WAVES) void traverse_kernel(TraverseArgs a) {
    // One static block, in this order: the compiler then knows every LDS
    // address, and a heap cell [j - 512] is j * 8 plus a constant that fits the
    // instruction's offset field.
    using Open = OpenList<H, deep_from(H)>;
    using Helped = LookAhead<WAVES - 1>;
    constexpr int S = (H + kWave - 1) / kWave;
    // cells of the final sort: all of them, and those sorted in LDS at once
    constexpr int kSortAll = H <= kWave ? kWave : 1 << (floor_log2(H - 1) + 1);
    constexpr int kSortLds = kSortAll > 1024 ? 1024 : kSortAll;
    // NEAR's lines in make_plan stand for room for the levels from 8 on and distances
    // of their own.  2 KB of it are idle at H = 512 and more: without them the same
    // times where the form stays the same, and where one more workgroup fits (250 000
    // rows, H = 512, 1000 queries, which then have helpers) rows of 40 floats 1.97 -> 1.69 ms,
    // of 64 1.51 -> 1.41, of 96 1.41 -> 1.28, of 128 1.26 -> 1.28.
    constexpr int kNearCells = !NEAR ? 0 : H == 2048 ? 1792 : 2 * H > 254 ? 2 * H - 254 : 0;
    constexpr int kListCells = Open::kLdsCells > kNearCells ? Open::kLdsCells : kNearCells;
    constexpr int kHeapCells = kListCells > kSortLds ? kListCells : kSortLds;
    // The table of recently marked rows in front of the bitmask: half the
    // size for the long lists, whose residency is bound by LDS (lists of 2048
    // and 4096 cells: 9 instead of 8 wavefronts per compute unit, 5 % faster
    // on 10 000 queries over 500 000 rows of 128 floats although the table
    // answers fewer tests; a quarter of the size is slower again, and
    // where LDS does not bound the residency the smaller table only costs).
    constexpr int kSeenLog2 =
        H >= 1024 && kSeenCacheLog2 > 0 ? kSeenCacheLog2 - 1 : kSeenCacheLog2;
    constexpr int kSeen = NEAR ? 4 : 1 << kSeenLog2;
    struct Lds {
        uint32_t seen_cache[kSeen];
        // a step's new rows, and then their distances
        int cand_id[WAVES > 1 ? 4 : kWave];
        float near_key[NEAR && WAVES == 1 ? kWave : 4];
        float query[DP8 ? query_floats(8 * DP8) : 4];
        int2 heap[kHeapCells];  // open list tail; the final sort reuses it
    };
    __shared__ __align__(16) Lds lds;
    __shared__ __align__(16) typename Helped::Slots slots;   // (WAVES > 1)
    // the query if its length is not known here, then NEAR's visited bits
    extern __shared__ __align__(16) float query_any_length[];
    const int lane = threadIdx.x & (kWave - 1);
    float *okey = reinterpret_cast<float *>(lds.heap);
    int *oval = reinterpret_cast<int *>(okey + kHeapCells);
    Open open;
    open.cells = lds.heap;
    int *cand_id = lds.cand_id;
    float *cand_key = NEAR ? lds.near_key : reinterpret_cast<float *>(lds.cand_id);
    float *qv = DP8 ? lds.query : query_any_length;
    const int dp = DP8 ? DP8 * 8 : a.dp;
    uint32_t *seen_cache = lds.seen_cache;
    const bool use_cache = a.n_storage <= (0xffff << kSeenLog2);
    const int deg = a.deg;
    uint32_t *seen = a.seen + (size_t)blockIdx.x * (size_t)a.slot_stride;
    uint32_t *near_bits =
        reinterpret_cast<uint32_t *>(query_any_length + (DP8 ? 0 : query_floats(dp)));
    Helped ahead{slots, -1, 0, 0};
    if constexpr (WAVES > 1) {
        const int wave = uni((int)(threadIdx.x / kWave));
        if (threadIdx.x < Helped::kJobs) Helped::put(slots.job[threadIdx.x], Helped::kIdle);
        __syncthreads();   // the only barrier
        if (wave > 0) {
            Helped::help(slots, lane, [&](int row, int, int *ids, float *dist) {
                // its neighbours, by lane, and the distances of those that are not
                // marked yet: a mark is never taken back, so whatever is new when
                // the node is popped is among them
                const int v = lane < deg ? a.adj[(size_t)row * deg + lane] : -1;
                ids[lane] = v;
                const bool maybe_new =
                    v >= 0 && !((Helped::get(near_bits[v >> 5]) >> (v & 31)) & 1u);
                eval_lanes<DP8, TWO>(a.storage, qv, maybe_new, v, dist, dp, lane);
            });
            return;
        }
    }
    // after the visited slice: the log of admitted candidates, then the
    // levels of the open list kept in device memory
    ResultLog log;
    log.entry = reinterpret_cast<int2 *>(seen + a.words_per_slot);
    log.capacity = ResultLog::capacity_for(H);
    open.deep = log.entry + ResultLog::capacity_for(H);

    for (int turn = 0;;) {
        const int q = next_query(a.work_counter, turn, a.batch, lane);
        if (q >= a.batch) {
            if constexpr (WAVES > 1) ahead.end(lane);
            break;
        }

        unsigned n_expand = 0, n_adj = 0, n_dist = 0, n_admit = 0;
#ifdef PA_PHASE_TIMERS
        unsigned long long phase[7] = {0, 0, 0, 0, 0, 0, 0};
#endif
        PA_TIMER_BEGIN();

        // fresh visited slice, query to LDS, empty lists
#ifndef PA_CLEAR_REPS  // tuning builds: the clearing repeated, to time it
#define PA_CLEAR_REPS 1
#endif
        for (int rep = 0; rep < PA_CLEAR_REPS; ++rep)
            for (int w = lane * 4; w < a.words_per_slot; w += kWave * 4)
                *reinterpret_cast<uint4 *>((NEAR ? near_bits : seen) + w) =
                    make_uint4(0, 0, 0, 0);
        for (int i = lane; i < dp; i += kWave)
            qv[query_slot(i, dp >> 3)] = a.query[(size_t)q * dp + i];
        for (int i = lane; i < kSeen; i += kWave) seen_cache[i] = 0xffffffffu;
        open.reset(lane);
        ResultKeys<S> res;
        res.init(H, lane);
        log.n = 0;
        // The clearing stores must have reached the cache level where the
        // atomic ORs are performed before the first OR is issued.  Only this
        // wavefront touches the slice, so waiting for its own stores is
        // enough; a device-scope fence here would write back and invalidate
        // caches once per query.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        wave_sync();

        // traverse_cpu.cpp:69-79: entries are marked and pushed on the open
        // list, in order.  An entry without a storage row has no adjacency
        // here; it is kept under the code -2-i (i = its position) so that it
        // is popped, and costs a step, like any other.
        const int64_t *eI = a.init_I + (size_t)q * a.n_init;
        const float *eD = a.init_D + (size_t)q * a.n_init;
        for (int base = 0; base < a.n_init; base += kWave) {
            const int i = base + lane;
            int u = -1, row = -1;
            float d = INFINITY;
            if (i < a.n_init) {
                const int64_t g = eI[i];
                d = eD[i];
                if (g >= 0 && g < a.n_nodes) {
                    u = (int)g;
                    row = (int)a.mapping[g];
                    if (row >= 0) {
                        if constexpr (NEAR)
                            atomicOr(&near_bits[row >> 5], 1u << (row & 31));
                        else
                            atomicOr(&seen[row >> 5], 1u << (row & 31));
                    }
                }
            }
            int value = row >= 0 ? row : u >= 0 ? -2 - i : -1;
            if constexpr (WAVES > 1) {
                if (base == 0) {
                    ahead.begin(lane);
                    for (int j = 0; j < WAVES - 1; ++j)
                        ahead.ask_lowest(list_key(d), value, lane);
                }
            }
            open.push_entries(__ballot(u >= 0), list_key(d), value, lane);
        }

        PA_TIMER(5);
        // traverse_cpu.cpp:82-136, software-pipelined.  The node a pop will
        // return is the root of the open list as it stands after the last
        // insert, so once a step's inserts are done the next step's node is
        // certain: its neighbours' visited bits are tested and set *before*
        // the pop (the atomics are in flight while the pop sifts).  If the
        // search ends at the next pop instead, the marks set for a node that
        // is never expanded are harmless: the slice is cleared per query.
        // That node's row of neighbour ids is requested still earlier, right
        // after the pop, for the root the pop leaves, and again only if an
        // insert put another node there: it travels while the rows are read
        // (one query, lists of 4096 cells, 5.49 -> 5.28 ms; 10 000, lists of
        // 768, 3.50 -> 3.47 ms; where the rows take the time it is the same).
        auto load_row = [&](int r) -> int {
            int row = -1;
            if (r >= 0 && lane < deg) row = a.adj[(size_t)r * deg + lane];
            return row;
        };
        // Returns the bitmask word before the OR; it is looked at only after
        // the pop.  Most neighbours of a node were seen a few steps ago: a
        // two-way LDS table of rows whose bit is known to be set answers for
        // them without going to memory.  Word r mod 1024 holds the 16-bit
        // tags r / 1024 of the two rows seen last (newest in the low half).
        // A row enters the table only after its atomic has been issued, so a
        // hit is always right; a miss (never seen, or displaced) asks the
        // bitmask, which is exact.
        auto test_and_set = [&](int v) -> uint32_t {
            uint32_t before = 0xffffffffu;
            if constexpr (NEAR) {
                if (v >= 0) before = atomicOr(&near_bits[v >> 5], 1u << (v & 31));
                return before;
            }
            if (v >= 0) {
                const int cell = v & (kSeen - 1);
                const uint32_t tag = (uint32_t)v >> kSeenLog2;
                const uint32_t ways = use_cache ? seen_cache[cell] : 0xffffffffu;
                if (!use_cache || ((ways & 0xffffu) != tag && (ways >> 16) != tag)) {
                    before = atomicOr(&seen[v >> 5], 1u << (v & 31));
                    if (use_cache) seen_cache[cell] = (ways << 16) | tag;
                }
            }
            return before;
        };
        // heap_update, traverse_cpu.cpp:25-39, in adjacency order: the lanes'
        // keys d and rows id; `value` is what the open list keeps of them
        auto admit = [&](int d, int id, int value) {
            unsigned long long todo = __ballot(d < res.worst);
            unsigned long long admitted = 0;
            while (todo) {
                const int j = __builtin_ctzll(todo);
                const int dj = __builtin_amdgcn_readlane(d, j);
                const int vj = __builtin_amdgcn_readlane(value, j);
                open.insert(dj, vj, lane, [&] { res.insert(dj, lane); });
                admitted |= 1ull << j;
                todo &= (todo - 1) & __ballot(d < res.worst);
            }
            if (admitted) {
                n_admit += __popcll(admitted);
                log.append(admitted, d, id, lane);
                if (log.nearly_full()) log.cut(res.worst, lane);
            }
        };
        if constexpr (WAVES > 1) {
            if (a.n_init == 0) ahead.begin(lane);
            for (int step = 0; step < a.max_iter; ++step) {
                const int u = open.root_val();
                if (u == -1 || open.root_key() >= res.worst) break;
                typename Helped::Found found;
                if (u >= 0) found = ahead.find(u & ~Helped::kAsked, lane);
                int popped_k, popped_v;
                open.pop(lane, popped_k, popped_v);
                n_expand += 1;
                if (u >= 0) {
                    n_adj += deg;
                    ahead.take(found, lane);
                    const int v = found.id;
                    uint32_t before = 0xffffffffu;
                    if (v >= 0) before = atomicOr(&near_bits[v >> 5], 1u << (v & 31));
                    ahead.ask(open.A.v, lane);
                    open.pop_finish();
                    const bool fresh = !((before >> (v & 31)) & 1u);
                    n_dist += __popcll(__ballot(fresh));
                    const int d = fresh ? list_key(found.dist) : Open::kInf;
                    // a neighbour that is before all of the list is next
                    int value = v;
                    if (__ballot(d < open.root_key()) && ahead.room()) {
                        const int best = ~wave_max_key(~d);
                        const int at = __builtin_ctzll(__ballot(d == best));
                        ahead.give(__builtin_amdgcn_readlane(v, at), lane);
                        value = lane == at ? v | Helped::kAsked : v;
                    }
                    admit(d, v, value);
                } else {
                    open.pop_finish();
                }
            }
            ahead.drain(lane);
        }
        int v = -1;
        uint32_t before = 0xffffffffu;
        if constexpr (WAVES == 1) {
            v = load_row(open.root_val());
            before = test_and_set(v);
        }
        for (int step = 0; WAVES == 1 && step < a.max_iter; ++step) {
            int uk, u;
            open.pop(lane, uk, u);
            const int likely = open.root_val();
            const int likely_row = load_row(likely);
            PA_TIMER(0);
            if (u == -1 || uk >= res.worst) break;
            n_expand += 1;
            bool popped = false;  // the pop has been finished
            if (u >= 0) {
                n_adj += deg;
                const bool fresh = !((before >> (v & 31)) & 1u);
                const unsigned long long mask = __ballot(fresh);
                const int n = __popcll(mask);
                PA_TIMER(2);
                if (n > 0) {
                    if (fresh) cand_id[lane_rank(mask)] = v;
                    wave_sync();
                    const int id = lane < n ? cand_id[lane] : -1;
                    wave_sync();
                    eval_rows<DP8, TWO>(a.storage, qv, cand_id, cand_key, n, dp, lane);
                    n_dist += n;
                    wave_sync();
                    PA_TIMER(3);
                    // levels of the open list in device memory: their pair
                    // was requested by the pop and has arrived with the rows
                    open.pop_finish();
                    popped = true;

                    admit(list_key(lane < n ? cand_key[lane] : INFINITY), id, id);
                    PA_TIMER(4);
                }
            }
            if (!popped) open.pop_finish();
            v = likely_row;
            const int root = open.root_val();
            if (root != likely) v = load_row(root);
            before = test_and_set(v);
            PA_TIMER(1);
        }

        // traverse_cpu.cpp:138-148: the entries compete for a result slot.  A
        // log value below -1 is the global id -2 - value of an entry, the
        // others are storage rows.
        for (int base = 0; base < a.n_init; base += kWave) {
            const int i = base + lane;
            int u = -1;
            float d = INFINITY;
            if (i < a.n_init) {
                const int64_t g = eI[i];
                d = eD[i];
                if (g >= 0 && g < a.n_nodes) u = (int)g;
            }
            const int dk = list_key(d);
            unsigned long long todo = __ballot(u >= 0 && dk < res.worst);
            unsigned long long admitted = 0;
            while (todo) {
                const int j = __builtin_ctzll(todo);
                todo &= todo - 1;
                const int dj = __builtin_amdgcn_readlane(dk, j);
                if (dj >= res.worst) continue;
                res.insert(dj, lane);
                admitted |= 1ull << j;
            }
            if (admitted) {
                log.append(admitted, dk, -2 - u, lane);
                if (log.nearly_full()) log.cut(res.worst, lane);
            }
        }

        // traverse_cpu.cpp:150-162: best first.  The set is read back from
        // the log — every entry below the maximum, and of those at the
        // maximum as many as make H — into the LDS the open list no longer
        // needs, padded to a power of two with +inf, and sorted there.
        wave_sync();
        ResultLog::settle();
        int n_below = 0;
        for (int base = 0; base < log.n; base += kWave) {
            const int i = base + lane;
            n_below += __popcll(__ballot(i < log.n && log.entry[i].x < res.worst));
        }
        // Stages of a bitonic network over okey / oval [0, n): merges of
        // `first_size` cells and up (2: a full sort; n: the last merge alone,
        // for cells that are bitonic already); `desc`: largest first.
        auto lds_sort = [&](int n, int first_size, bool desc) {
            for (int size = first_size; size <= n; size <<= 1) {
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    for (int t = lane; t < (n >> 1); t += kWave) {
                        const int i = ((t & ~(stride - 1)) << 1) | (t & (stride - 1));
                        const int j = i | stride;
                        const float ki = okey[i], kj = okey[j];
                        const int vi = oval[i], vj = oval[j];
                        const bool gt = ki > kj || (ki == kj && vi > vj);
                        const bool lt = ki < kj || (ki == kj && vi < vj);
                        if ((((i & size) == 0) != desc) ? gt : lt) {
                            okey[i] = kj, oval[i] = vj;
                            okey[j] = ki, oval[j] = vi;
                        }
                    }
                    wave_sync();
                }
            }
        };
        int64_t *oI = a.out_I + (size_t)q * a.k;
        float *oD = a.out_D + (size_t)q * a.k;
        if constexpr (kSortAll <= kSortLds) {
            for (int i = lane; i < a.sort_n; i += kWave)
                okey[i] = INFINITY, oval[i] = -1;
            wave_sync();
            int at_below = 0, at_worst = n_below;
            for (int base = 0; base < log.n; base += kWave) {
                const int i = base + lane;
                int2 e = make_int2(0x7fffffff, -1);
                if (i < log.n) e = log.entry[i];
                const bool below = i < log.n && e.x < res.worst;
                const bool tie = i < log.n && e.x == res.worst;
                const unsigned long long mb = __ballot(below), mt = __ballot(tie);
                int place = -1;
                if (below) place = at_below + lane_rank(mb);
                if (tie) place = at_worst + lane_rank(mt);
                if (place >= 0 && place < H) {
                    okey[place] = key_to_float(e.x);
                    oval[place] = e.y < -1 ? -2 - e.y : a.gid[e.y];
                }
                at_below += __popcll(mb);
                at_worst += __popcll(mt);
            }
            wave_sync();
            lds_sort(a.sort_n, 2, false);
            for (int i = lane; i < a.k; i += kWave) {
                oI[i] = (int64_t)oval[i];
                oD[i] = okey[i];
            }
        } else {
            // The longest lists sort in two halves of kSortLds cells, so that
            // the sort does not decide the size of the LDS block (and with it
            // how many wavefronts a compute unit holds).  The set is
            // compacted at the head of the log (in log order: a write lands
            // on an entry already read), as (distance, id); the first half is
            // sorted ascending and the second descending through LDS; one
            // exchange between the halves in the log leaves every cell of the
            // first below every cell of the second and both bitonic; each is
            // then merged in LDS and written out.
            static_assert(kSortAll == 2 * kSortLds, "two halves");
            static_assert(ResultLog::capacity_for(H) >= kSortAll, "the log holds them");
            int m = 0, ties_left = H - n_below;
            for (int base = 0; base < log.n; base += kWave) {
                const int i = base + lane;
                int2 e = make_int2(0x7fffffff, -1);
                if (i < log.n) e = log.entry[i];
                const bool below = i < log.n && e.x < res.worst;
                const bool tie = i < log.n && e.x == res.worst;
                const unsigned long long mt = __ballot(tie);
                const bool keep = below || (tie && lane_rank(mt) < ties_left);
                const unsigned long long mk = __ballot(keep);
                if (keep) {
                    const int id = e.y < -1 ? -2 - e.y : a.gid[e.y];
                    log.entry[m + lane_rank(mk)] =
                        make_int2(__float_as_int(key_to_float(e.x)), id);
                }
                m += __popcll(mk);
                ties_left -= min(ties_left, (int)__popcll(mt));
            }
            ResultLog::settle();
            auto load_half = [&](int half) {
                for (int i = lane; i < kSortLds; i += kWave) {
                    const int at = half * kSortLds + i;
                    int2 e = make_int2(__float_as_int(INFINITY), -1);
                    if (at < m) e = log.entry[at];
                    okey[i] = __int_as_float(e.x), oval[i] = e.y;
                }
                wave_sync();
            };
            for (int half = 0; half < 2; ++half) {
                load_half(half);
                lds_sort(kSortLds, 2, half == 1);
                for (int i = lane; i < kSortLds; i += kWave)
                    log.entry[half * kSortLds + i] =
                        make_int2(__float_as_int(okey[i]), oval[i]);
                wave_sync();
            }
            ResultLog::settle();
            m = kSortAll;  // both halves are whole now, +inf cells included
            for (int i = lane; i < kSortLds; i += kWave) {
                const int2 x = log.entry[i], y = log.entry[kSortLds + i];
                const float kx = __int_as_float(x.x), ky = __int_as_float(y.x);
                if (kx > ky || (kx == ky && x.y > y.y)) {
                    log.entry[i] = y;
                    log.entry[kSortLds + i] = x;
                }
            }
            ResultLog::settle();
            for (int half = 0; half < 2; ++half) {
                load_half(half);
                lds_sort(kSortLds, kSortLds, false);
                for (int i = lane; i < kSortLds; i += kWave) {
                    const int r = half * kSortLds + i;
                    if (r < a.k) {
                        oI[r] = (int64_t)oval[i];
                        oD[r] = okey[i];
                    }
                }
                wave_sync();
            }
        }
        wave_sync();

        if (a.counters && lane == 0) {
            atomicAdd(&a.counters[0], (unsigned long long)n_expand);
            atomicAdd(&a.counters[1], (unsigned long long)n_adj);
            atomicAdd(&a.counters[2], (unsigned long long)n_dist);
            atomicAdd(&a.counters[3], (unsigned long long)n_admit);
            atomicAdd(&a.counters[4], (unsigned long long)a.k);
#ifdef PA_PHASE_TIMERS
            PA_TIMER(6);
            for (int i = 0; i < 7; ++i) atomicAdd(&a.counters[5 + i], phase[i]);
#endif
        }
    }
}

// ---- graph preparation ----------------------------------------------------------

__global__ void fill_i32(int32_t *p, int64_t n, int32_t value) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

__global__ void invert_mapping(const int64_t *mapping, int64_t n_nodes,
                               int64_t n_storage, int32_t *gid,
                               int32_t *status) {
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_nodes) return;
    const int64_t row = mapping[g];
    if (row < 0) return;
    if (row >= n_storage) {
        atomicOr(status, 1);
        return;
    }
    if (atomicExch(&gid[row], (int32_t)g) != -1) atomicOr(status, 1);
}

// One wavefront per storage row; lane i looks at entry i of the node's row.
__global__ __launch_bounds__(256) void build_rows(
    const int64_t *indptr, const int64_t *indices, const int64_t *mapping,
    int64_t n_nodes, int64_t n_storage, int64_t nnz, int deg,
    const int32_t *gid, int32_t *adj, int32_t *status) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t r = (int64_t)blockIdx.x * (blockDim.x / kWave) +
                      (threadIdx.x / kWave);
    if (r >= n_storage) return;
    const int g = gid[r];
    int keep_row = -1;
    int n_valid = 0;
    if (g < 0) {
        if (lane == 0) atomicOr(status, 1);
    } else {
        const int64_t lo = indptr[g];
        int64_t len = indptr[g + 1] - lo;
        if (len > deg) {
            if (lane == 0) atomicOr(status, 2);
            len = deg;
        }
        if (len < 0) len = 0;
        // a row that does not lie inside `indices` is reported and read as
        // empty: nothing outside the array is ever touched
        if (lo < 0 || lo > nnz || len > nnz - lo) {
            if (lane == 0) atomicOr(status, 8);
            len = 0;
        }
        int64_t e = -1;
        if (lane < len) e = indices[lo + lane];
        const unsigned long long neg = __ballot(lane < len && e < 0);
        n_valid = neg ? __builtin_ctzll(neg) : (int)len;
        bool ok = lane < n_valid;
        if (ok && e >= n_nodes) {
            atomicOr(status, 4);
            ok = false;
        }
        int row = ok ? (int)mapping[e] : -1;
        if (row >= n_storage) row = -1;
        if (row == r) row = -1;
        // an entry equal to an earlier one of the row is dropped
        for (int j = 0; j < n_valid; ++j) {
            const int other = __builtin_amdgcn_readlane(row, j);
            if (j < lane && other == row) row = -1;
        }
        keep_row = row;
    }
    const unsigned long long kept = __ballot(keep_row >= 0);
    const int n_kept = __popcll(kept);
    int32_t *out = adj + r * deg;
    if (keep_row >= 0) out[lane_rank(kept)] = keep_row;
    if (lane >= n_kept && lane < deg) out[lane] = -1;
}

// ---- scratch for callers that cannot allocate -----------------------------------
//
// pa_traverse_static runs the search in this array instead of a caller's
// workspace.  Every GPU the library is used on holds its own copy at its own
// address; host code never uses the array's name as a pointer, only the
// address hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) unsigned char scratch[PA_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;

// Device address of `scratch` on the current device, looked up once per device.
int static_scratch(unsigned char **out) {
    static std::mutex mutex;
    static unsigned char *known[kMaxDevices] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return PA_E_RANGE;
    std::lock_guard<std::mutex> guard(mutex);
    if (!known[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!ptr) return PA_E_NULL;
        known[dev] = static_cast<unsigned char *>(ptr);
    }
    *out = known[dev];
    return PA_OK;
}

// ---- host side --------------------------------------------------------------------

int round_up(int64_t x, int64_t m) { return (int)(((x + m - 1) / m) * m); }

int next_pow2(int x) {
    int p = 1;
    while (p < x) p <<= 1;
    return p;
}

typedef void (*TraverseFn)(TraverseArgs);

// more than five wavefronts per SIMD have measured slower on every instance
// that fits them (the SIMDs' issue slots are the bound)
#ifndef PA_MAX_WAVES_PER_CU
#define PA_MAX_WAVES_PER_CU 20
#endif
constexpr int kMaxWavesPerCu = PA_MAX_WAVES_PER_CU;
constexpr int kStaticLds = 20 << 10;   // no instance has more static LDS
constexpr int kHelped = 4;   // wavefronts of a query when there are few queries
constexpr int64_t kTwoRowsBytes = 160ll << 20;   // see make_plan

template <int H, bool NEAR, bool TWO, int WAVES>
TraverseFn pick_dp(int dp) {
    if (TWO) return dp == 128 ? traverse_kernel<H, 16, NEAR, true, WAVES> : nullptr;
    switch (dp) {
        case 32: return traverse_kernel<H, 4, NEAR, false, WAVES>;
        case 64: return traverse_kernel<H, 8, NEAR, false, WAVES>;
        case 128: return NEAR ? nullptr : traverse_kernel<H, 16, false, false, 1>;
        default: return traverse_kernel<H, 0, NEAR, false, WAVES>;
    }
}

template <bool NEAR, bool TWO, int WAVES = 1>
TraverseFn pick_kernel(int H, int dp) {
    switch (H) {
        case 16: return pick_dp<16, NEAR, TWO, WAVES>(dp);
        case 32: return pick_dp<32, NEAR, TWO, WAVES>(dp);
        case 48: return pick_dp<48, NEAR, TWO, WAVES>(dp);
        case 64: return pick_dp<64, NEAR, TWO, WAVES>(dp);
        case 96: return pick_dp<96, NEAR, TWO, WAVES>(dp);
        case 128: return pick_dp<128, NEAR, TWO, WAVES>(dp);
        case 192: return pick_dp<192, NEAR, TWO, WAVES>(dp);
        case 256: return pick_dp<256, NEAR, TWO, WAVES>(dp);
        case 384: return pick_dp<384, NEAR, TWO, WAVES>(dp);
        case 512: return pick_dp<512, NEAR, TWO, WAVES>(dp);
        case 1024: return pick_dp<1024, NEAR, TWO, WAVES>(dp);
        case 2048: return pick_dp<2048, NEAR, TWO, WAVES>(dp);
        default: return nullptr;
    }
}

// Wavefronts (workgroups of one) of `fn` the current device holds at once, and
// in *max_lds what LDS it gives one workgroup.
int residency(TraverseFn fn, int threads, int lds_bytes, int64_t *slots, int *max_lds) {
    struct Known {
        int cus, per_cu, max_lds;
    };
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    // the residency of a (device, kernel, LDS size) never changes
    static std::mutex mutex;
    static std::map<std::tuple<int, const void *, int>, Known> known;
    std::lock_guard<std::mutex> guard(mutex);
    const auto key = std::make_tuple(dev, reinterpret_cast<const void *>(fn), lds_bytes);
    auto it = known.find(key);
    if (it == known.end()) {
        Known k = {0, 0, 0};
        e = hipDeviceGetAttribute(&k.cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e == hipSuccess)
            e = hipDeviceGetAttribute(&k.max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
        if (e == hipSuccess)
            e = workgroups_per_cu(reinterpret_cast<const void *>(fn), dev, threads, lds_bytes,
                                  &k.per_cu);
        if (e != hipSuccess) return (int)e;
        // sizes of NEAR follow the index: a few stay
        if (known.size() > 4096) known.clear();
        it = known.emplace(key, k).first;
    }
    *slots = (int64_t)it->second.per_cu * it->second.cus;
    *max_lds = it->second.max_lds;
    if (it->second.per_cu > kMaxWavesPerCu) *slots = (int64_t)kMaxWavesPerCu * it->second.cus;
    return PA_OK;
}

struct Plan {
    int H, sort_n, lds_bytes, n_slots, words_per_slot, slot_stride, threads;
    size_t workspace_bytes;
    TraverseFn fn;
    bool near_bits;
};

// `beside`: queries of other launches at the same time.  It decides about the
// form alone; the workspace is the same.
int make_plan(int64_t n_storage, int64_t batch, int64_t beside, int dp, int ef_total, Plan *p) {
    if (n_storage <= 0 || batch < 0 || beside < 0) return PA_E_SHAPE;
    if (n_storage >= (1ll << 31)) return PA_E_RANGE;
    if (dp <= 0 || dp % 8) return PA_E_DIM;
    if (ef_total < 1 || ef_total > PA_MAX_EF_TOTAL) return PA_E_EF;
    p->H = pa_heap_size(ef_total);
    p->sort_n = next_pow2(p->H < kWave ? kWave : p->H);
    // dynamic LDS: the query when its length has no specialised kernel (the
    // rest is static in the kernel)
    p->lds_bytes = (dp == 32 || dp == 64 || dp == 128) ? 0 : query_floats(dp) * 4;
#ifdef PA_EXTRA_LDS  // tuning builds: lower the residency without touching code
    p->lds_bytes += PA_EXTRA_LDS;
#endif
    p->near_bits = false;
    p->threads = kWave;
    p->fn = dp == 128 ? pick_kernel<false, true>(p->H, dp) : pick_kernel<false, false>(p->H, dp);
    if (!p->fn) return PA_E_EF;
    int64_t slots = 0;
    int max_lds = 0;
    const int rc = residency(p->fn, kWave, p->lds_bytes, &slots, &max_lds);
    if (rc != PA_OK) return rc;
    // 128-float rows: two passes of reads in flight per wavefront, or one and five
    // wavefronts per SIMD instead of three.  Two where the queries all run at
    // once; beyond that one, if it still has them all at once and two would leave
    // most of a second round empty, where the rows do not stay in cache, or
    // with lists of 4096 cells (ten instead of eight wavefronts).  Measured, two passes /
    // one, ms.  250 000 rows of a million of 768 floats: H = 128, 3500 queries 1.20 / 1.10,
    // 10 000 2.59 / 2.68, 40 000 9.60 / 9.66; H = 256, 6000 2.95 / 3.07, 40 000 17.1 / 17.4;
    // H = 512, 10 000 10.5 / 10.8.  Rows of a mixture in 128 dimensions, which share more of
    // their neighbours: 350 000, H = 192, 5000 1.60 / 1.41, 40 000 9.39 / 8.48; 500 000, H =
    // 256, 10 000 3.61 / 3.16, 40 000 12.1 / 9.85; 250 000, H = 2048, 10 000 23.7 / 21.8; but one
    // is the better on fewer of these too from H = 128 on: 75 000, H = 256, 10 000 2.42 / 2.16;
    // 250 000, H = 128 1.78 / 1.75, H = 256 2.84 / 2.60 (H = 64 1.35 / 1.39).
    if (dp == 128 && batch > slots - beside) {
        const TraverseFn one = pick_kernel<false, false>(p->H, dp);
        int64_t one_slots = 0;
        const int one_rc = residency(one, kWave, p->lds_bytes, &one_slots, &max_lds);
        if (one_rc != PA_OK) return one_rc;
        const bool short_round =
            batch <= one_slots - beside && batch <= 4 * slots / 3 - beside;
        // (where LDS holds no more of them than of the other form, as with lists
        // of 2048 cells, two: 500 000 rows, 40 000 queries 37.8 / 38.0)
        if (one_slots > slots &&
            (short_round || n_storage * 512 > kTwoRowsBytes || p->H > 1024))
            p->fn = one, slots = one_slots;
    }
    p->n_slots = (int)(slots < batch ? slots : batch);
    if (p->n_slots < 1) p->n_slots = 1;
    p->words_per_slot = round_up((n_storage + 31) / 32, kSlotAlignWords);
    // a slot: the visited slice, the log of admitted candidates, the levels
    // of the open list that are kept in device memory (8 bytes an entry or cell)
    p->slot_stride = p->words_per_slot + 2 * ResultLog::capacity_for(p->H) +
                     round_up(2 * open_list_deep_cells(p->H, deep_from(p->H)), kWave);
    p->workspace_bytes =
        kWorkCounterBytes + (size_t)p->n_slots * p->slot_stride * 4;
    // The visited bits in LDS as long as every query, those of launches beside
    // this one too, still has its wavefront at once: a test there is one LDS
    // operation where it was a table look-up and a trip to L2 or beyond for the
    // atomic.  (One word of table: a build for tests of the paths behind it.)
    // Measured without helpers on 250 000 rows (31 KB, 1024 queries fit), far / near, us:
    // 128 floats, H = 128, one query 221 / 205, 37 382 / 378, 1024 516 / 493; H = 192, 512 686 /
    // 610; 64 floats, H = 384, 37 929 / 885; 40 floats, H = 256, 1000 1373 / 1256; 500 000 rows
    // of 128, H = 1024, 512 2416 / 2182.
    // Where only the other form has all queries at once, that one (whole searches in
    // two halves, far / near, ms: 100 000 rows of 64 floats, H = 512, 2 x 1500 2.16 / 2.34,
    // 2 x 2000 2.27 / 2.74; 75 000 of 40, H = 128, 2 x 2000 0.83 / 0.95; but 100 000 of 128, H =
    // 64, 2 x 2000 0.64 / 0.60).  Where neither has, near bits if they take no query's
    // place (20 000 rows, 10 000 queries: 128 floats, H = 64 0.86 / 0.74, H = 512 3.54 / 3.35; 32
    // floats, H = 256 1.84 / 1.72), or up to a third of them and each launch runs at once
    // (2 x 2500: 50 000 rows of 40 floats, H = 256 1.66 / 1.53; 75 000 of 128, H = 256 1.66 /
    // 1.52; at the end of it the other form is the better: 75 000 of 64, H = 256 1.42 / 1.55).
    const int64_t near_lds = p->lds_bytes + (int64_t)p->words_per_slot * 4;
    if (kSeenCacheLog2 > 0 && near_lds + kStaticLds <= max_lds) {
        const TraverseFn near_fn =
            dp == 128 ? pick_kernel<true, true>(p->H, dp) : pick_kernel<true, false>(p->H, dp);
        int64_t near_slots = 0;
        const int near_rc = residency(near_fn, kWave, (int)near_lds, &near_slots, &max_lds);
        if (near_rc != PA_OK) return near_rc;
        const bool near_fits = batch <= near_slots - beside;
        const bool far_fits = batch <= slots - beside;
        if (near_fits ||
            (!far_fits && (near_slots >= slots ||
                           (batch <= near_slots && 3 * near_slots >= 2 * slots)))) {
            p->fn = near_fn, p->lds_bytes = (int)near_lds;
            p->near_bits = true;
        }
        // With three helpers as long as every query, those of launches beside this
        // one too, has its four wavefronts at once.  Measured, without / with, us:
        // 250 000 rows of a million of 768 floats, dp = 128, H = 128, one query 262 / 201
        // (the median of 60), 37 418 / 333, 1024 510 / 419; H = 192, 37 592 / 459; H = 256, 512
        // 820 / 650, 1024 843 / 754; H = 1024, 37 3198 / 2552, 512 (the most that fit) 3348 /
        // 2765; rows of 64 floats, H = 384, 100 1121 / 1033; of 40, H = 256, 1000 1256 / 946.
        // (Seven helpers, H = 128, one query: the same; H = 256, 1024: 905 where three
        // take 770.)  An expansion over rows of 32 floats is list work, and in lists
        // of 768 cells and more how much of it depends on the rows: 25 000 of 100 000 in 64
        // clusters, H = 384, 1000 660 / 776, H = 512 852 / 996, H = 1024 1748 / 2010; 250 000 of a
        // wider mixture, H = 384, 500 1539 / 1348, H = 1024, 700 3043 / 2627.  Up to H = 256
        // helpers are the faster on both (128 on the first 388 / 370, 1000 on the second
        // 965 / 830).
        if (near_fits && (dp > 32 || p->H <= 256)) {
            const TraverseFn helped_fn = dp == 128 ? pick_kernel<true, true, kHelped>(p->H, dp)
                                                   : pick_kernel<true, false, kHelped>(p->H, dp);
            int64_t helped_slots = 0;
            const int helped_rc = residency(helped_fn, kHelped * kWave, (int)near_lds,
                                            &helped_slots, &max_lds);
            if (helped_rc != PA_OK) return helped_rc;
            if (batch <= helped_slots - beside)
                p->fn = helped_fn, p->threads = kHelped * kWave;
        }
    }
    return PA_OK;
}

}  // namespace

extern "C" int pa_heap_size(int ef_search) {
    static const int ladder[] = {16,  32,  48,  64,  96,   128,
                                 192, 256, 384, 512, 1024, 2048};
    for (int h : ladder)
        if (ef_search <= h) return h;
    return -1;
}

extern "C" const char *pa_error_string(int code) {
    if (code > 0) return hipGetErrorString((hipError_t)code);
    switch (code) {
        case PA_OK: return "ok";
        case PA_E_NULL: return "a required pointer is null";
        case PA_E_SHAPE: return "a size is negative or inconsistent";
        case PA_E_DIM: return "vector length must be a multiple of 8";
        case PA_E_NEIGHBORS: return "n_neighbors must be in 1..64";
        case PA_E_EF: return "beam * ef must be in 1..2048";
        case PA_E_WORKSPACE: return "workspace too small or not 256-byte aligned";
        case PA_E_GRAPH: return "malformed graph (see status word)";
        case PA_E_LEAVES: return "n_leaves must be a multiple of 32";
        case PA_E_CHUNK: return "batch must be a multiple of chunk_size";
        case PA_E_RANGE: return "an id does not fit 31 bits";
        case PA_E_STATIC:
            return "index too large for the static scratch of pa_traverse_static";
        default: return "unknown error";
    }
}

extern "C" int pa_graph_prepare(const int64_t *indptr, const int64_t *indices,
                                const int64_t *mapping, int64_t n_nodes,
                                int64_t n_storage, int64_t nnz,
                                int n_neighbors, int32_t *adj, int32_t *gid,
                                int32_t *status, void *stream_) {
    if (n_nodes <= 0 || n_storage <= 0 || n_storage > n_nodes || nnz < 0)
        return PA_E_SHAPE;
    if (!indptr || !indices || !mapping || !adj || !gid || !status)
        return PA_E_NULL;
    if (n_nodes >= (1ll << 31)) return PA_E_RANGE;
    if (n_neighbors < 1 || n_neighbors > PA_MAX_NEIGHBORS) return PA_E_NEIGHBORS;
    hipStream_t stream = (hipStream_t)stream_;
    const int T = 256;
    fill_i32<<<1, 1, 0, stream>>>(status, 1, 0);
    fill_i32<<<(unsigned)((n_storage + T - 1) / T), T, 0, stream>>>(gid, n_storage, -1);
    invert_mapping<<<(unsigned)((n_nodes + T - 1) / T), T, 0, stream>>>(
        mapping, n_nodes, n_storage, gid, status);
    const int rows_per_block = T / kWave;
    build_rows<<<(unsigned)((n_storage + rows_per_block - 1) / rows_per_block), T,
                 0, stream>>>(indptr, indices, mapping, n_nodes, n_storage,
                              nnz, n_neighbors, gid, adj, status);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    int32_t host_status = 0;
    e = hipMemcpyAsync(&host_status, status, sizeof(int32_t),
                       hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return (int)e;
    return host_status ? PA_E_GRAPH : PA_OK;
}

extern "C" int pa_traverse_plan(int64_t n_storage, int64_t batch, int dp,
                                int ef_total, int *n_slots,
                                size_t *workspace_bytes) {
    Plan p;
    const int rc = make_plan(n_storage, batch, 0, dp, ef_total, &p);
    if (rc != PA_OK) return rc;
    if (n_slots) *n_slots = p.n_slots;
    if (workspace_bytes) *workspace_bytes = p.workspace_bytes;
    return PA_OK;
}

extern "C" int pa_traverse_form(int64_t n_storage, int64_t batch, int64_t beside, int dp,
                                int ef_total, int *near_bits) {
    Plan p;
    const int rc = make_plan(n_storage, batch, beside, dp, ef_total, &p);
    if (rc != PA_OK) return rc;
    if (near_bits) *near_bits = p.near_bits;
    return PA_OK;
}

extern "C" int pa_traverse_wavefronts(int64_t n_storage, int64_t batch, int64_t beside, int dp,
                                      int ef_total, int *wavefronts) {
    Plan p;
    const int rc = make_plan(n_storage, batch, beside, dp, ef_total, &p);
    if (rc != PA_OK) return rc;
    if (wavefronts) *wavefronts = p.threads / kWave;
    return PA_OK;
}

namespace {

// Checks and launch shared by pa_traverse and pa_traverse_static.  With
// `fit_slots` the number of wavefronts is lowered to what the workspace holds
// (at least min(batch, kMinStaticSlots), else PA_E_STATIC); without it a
// workspace smaller than the plan's is an error.
constexpr int kMinStaticSlots = 256;

int launch_traverse(int64_t *out_I, float *out_D, const int32_t *adj,
                    const int32_t *gid, const int64_t *mapping,
                    const float *storage, const float *query,
                    const int64_t *init_I, const float *init_D, int64_t batch,
                    int64_t beside, int64_t n_nodes, int64_t n_storage, int dp,
                    int n_init, int beam, int ef, int n_neighbors, void *workspace,
                    size_t workspace_bytes, bool fit_slots, uint64_t *counters,
                    void *stream_) {
    if (batch < 0 || n_nodes <= 0 || n_init < 0 || beam < 1 || ef < 1)
        return PA_E_SHAPE;
    if (n_nodes >= (1ll << 31) || batch >= (1ll << 31)) return PA_E_RANGE;
    if (n_neighbors < 1 || n_neighbors > PA_MAX_NEIGHBORS) return PA_E_NEIGHBORS;
    if ((int64_t)beam * ef > PA_MAX_EF_TOTAL) return PA_E_EF;
    Plan p;
    const int rc = make_plan(n_storage, batch, beside, dp, beam * ef, &p);
    if (rc != PA_OK) return rc;
    if (batch == 0) return PA_OK;
    if (!out_I || !out_D || !adj || !gid || !mapping || !storage || !query ||
        !workspace || (n_init > 0 && (!init_I || !init_D)))
        return PA_E_NULL;
    if (fit_slots) {
        const size_t slot_bytes = (size_t)p.slot_stride * 4;
        const size_t fit = workspace_bytes < kWorkCounterBytes
                               ? 0
                               : (workspace_bytes - kWorkCounterBytes) / slot_bytes;
        const int64_t need = batch < kMinStaticSlots ? batch : kMinStaticSlots;
        if ((int64_t)fit < need) return PA_E_STATIC;
        if ((size_t)p.n_slots > fit) p.n_slots = (int)fit;
    } else if (workspace_bytes < p.workspace_bytes) {
        return PA_E_WORKSPACE;
    }
    if (reinterpret_cast<uintptr_t>(workspace) % 256) return PA_E_WORKSPACE;

    TraverseArgs a;
    a.out_I = out_I, a.out_D = out_D;
    a.adj = adj, a.gid = gid, a.mapping = mapping;
    a.storage = storage, a.query = query;
    a.init_I = init_I, a.init_D = init_D;
    a.work_counter = p.n_slots < batch ? reinterpret_cast<int *>(workspace) : nullptr;
    a.seen = reinterpret_cast<uint32_t *>(
        reinterpret_cast<unsigned char *>(workspace) + kWorkCounterBytes);
    a.counters = reinterpret_cast<unsigned long long *>(counters);
    a.batch = (int)batch, a.n_nodes = (int)n_nodes, a.n_storage = (int)n_storage;
    a.dp = dp, a.n_init = n_init, a.k = beam * ef, a.H = p.H;
    a.deg = n_neighbors;
    // traverse_cpu.cpp:18,82
    a.max_iter = 2 * beam * ef < 1024 ? 2 * beam * ef : 1024;
    a.words_per_slot = p.words_per_slot, a.sort_n = p.sort_n;
    a.slot_stride = p.slot_stride;

    hipStream_t stream = (hipStream_t)stream_;
    if (a.work_counter) reset_work_counter<<<1, 1, 0, stream>>>(a.work_counter);
    p.fn<<<p.n_slots, p.threads, p.lds_bytes, stream>>>(a);
    return (int)hipGetLastError();
}

}  // namespace

extern "C" int pa_traverse(int64_t *out_I, float *out_D, const int32_t *adj,
                           const int32_t *gid, const int64_t *mapping,
                           const float *storage, const float *query,
                           const int64_t *init_I, const float *init_D,
                           int64_t batch, int64_t n_nodes, int64_t n_storage,
                           int dp, int n_init, int beam, int ef,
                           int n_neighbors, void *workspace,
                           size_t workspace_bytes, uint64_t *counters,
                           void *stream_) {
    return launch_traverse(out_I, out_D, adj, gid, mapping, storage, query,
                           init_I, init_D, batch, 0, n_nodes, n_storage, dp,
                           n_init, beam, ef, n_neighbors, workspace,
                           workspace_bytes, false, counters, stream_);
}

extern "C" int pa_traverse_beside(int64_t *out_I, float *out_D, const int32_t *adj,
                                  const int32_t *gid, const int64_t *mapping,
                                  const float *storage, const float *query,
                                  const int64_t *init_I, const float *init_D,
                                  int64_t batch, int64_t beside, int64_t n_nodes,
                                  int64_t n_storage, int dp, int n_init, int beam, int ef,
                                  int n_neighbors, void *workspace, size_t workspace_bytes,
                                  uint64_t *counters, void *stream_) {
    return launch_traverse(out_I, out_D, adj, gid, mapping, storage, query,
                           init_I, init_D, batch, beside, n_nodes, n_storage, dp,
                           n_init, beam, ef, n_neighbors, workspace,
                           workspace_bytes, false, counters, stream_);
}

extern "C" int pa_traverse_static(int64_t *out_I, float *out_D,
                                  const int32_t *adj, const int32_t *gid,
                                  const int64_t *mapping, const float *storage,
                                  const float *query, const int64_t *init_I,
                                  const float *init_D, int64_t batch,
                                  int64_t n_nodes, int64_t n_storage, int dp,
                                  int n_init, int beam, int ef, int n_neighbors,
                                  uint64_t *counters, void *stream_) {
    unsigned char *ws = nullptr;
    const int rc = static_scratch(&ws);
    if (rc != PA_OK) return rc;
    // The work counter is set by a kernel, the visited slices and the result
    // values are cleared by the search itself, per query: nothing of an
    // earlier call is read.
    return launch_traverse(out_I, out_D, adj, gid, mapping, storage, query,
                           init_I, init_D, batch, 0, n_nodes, n_storage, dp,
                           n_init, beam, ef, n_neighbors, ws,
                           PA_STATIC_SCRATCH_BYTES, true, counters, stream_);
}
