// Full-dimension refine on the device, for gfx950.
//
// The reference refines the device stage's candidates on the host
// (extension/traverse_cpu.cpp:261-369): per query two searches of
// traverse_cpu_kernel (:12-163) that share one visited set — first on the
// sampled subgraph, two expansions at most, from the candidates, whose
// distances over the first d_principle coordinates are completed to the full
// dimension in place (:42-62); then on the full graph from what the first one
// kept.  Here one wavefront runs both searches of a query, with the lists of
// the subgraph traversal (search_lists.h): the same array heap cell for cell,
// the same eight-accumulator distances bit for bit, an exact visited set (an LDS
// table; a node that finds its bucket full has a bit in the wavefront's slice of
// a pooled bitmask), kept across the two searches.  Rows are d_model floats; a
// quad of lanes streams a row sixteen 32-byte groups at a time.  In launches
// whose queries all run at once three more wavefronts read a query's rows with
// the first, 32 groups at a time; with a compute unit to a query, seven more read
// the rows of the nodes it is about to expand.
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

struct RefineArgs {
    int64_t *out_I;          // [batch, k]
    float *out_D;
    int64_t *buf_I;          // [batch, n_buffers]
    float *buf_D;
    const int64_t *init_I;   // [batch, n_init]
    float *init_D;           // completed in place
    const int32_t *sub_adj;  // prepared subgraph: rows of sampled-node ranks
    const int32_t *sub_gid;  // rank -> node
    const int64_t *sub_mapping;  // node -> rank or -1
    const int32_t *full_adj; // prepared full graph: rows of nodes
    const float *storage;    // [n_nodes, d]
    const float *query;      // [batch, d]
    uint32_t *seen;
    int *work_counter;
    unsigned long long *counters;
    int batch, n_nodes, d, dp, n_init, n_buffers, k, H;
    int sub_deg, full_deg, sub_iter, full_iter;
    int words_per_slot, slot_stride, sort_n;
};

__global__ void reset_refine_counter(int *counter) { *counter = 0; }

// Optional per-phase cycle tally for tuning builds (-DPA_PHASE_TIMERS): adds
// eight words after the six work counters.
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

// Squared L2 over the coordinates [from, d) between the query (LDS) and the
// rows listed in cand_id[0..n), written to cand_key: 16 rows per pass, four
// lanes per row; the accumulators start at zero at `from`
// (extension/inc/distance.h:31-55 called with an offset, traverse_cpu.cpp:56-59).
// Rows are in the interleaved layout of pa_rows_prepare.  The WAVES wavefronts
// of a workgroup take 16 rows each in turn.
template <int WAVES, int CHUNK>
__device__ __forceinline__ void eval_rows_from(const float *__restrict__ storage,
                                               const float *qv, const int *cand_id,
                                               float *cand_key, int n, int d,
                                               int from, int lane, int wave) {
    const int quad = lane >> 2, part = lane & 3;
    const int groups = d >> 3;
    const float2 *qrun =
        reinterpret_cast<const float2 *>(qv) + part * query_run(groups);
    for (int base = wave * kRowsPerPass; base < n; base += WAVES * kRowsPerPass) {
        const int c = base + quad;
        const bool active = c < n;
        const float *row = storage;
        if (active) row = storage + (size_t)cand_id[c] * (size_t)d;
        const float s = quad_square_dist_long<CHUNK>(row, qrun, groups, from >> 3,
                                                     part, active);
        if (active && part == 0) cand_key[c] = s;
    }
}

// The same for the rows of the lanes that `wanted` names, by one wavefront; the
// distance of lane l's row to dist[l].
template <int CHUNK>
__device__ __forceinline__ void eval_lanes_from(const float *__restrict__ storage,
                                                const float *qv, bool wanted, int id,
                                                float *dist, int d, int from, int lane) {
    const LaneRows rows(wanted, id, lane);
    const int quad = lane >> 2, part = lane & 3;
    const int groups = d >> 3;
    const float2 *qrun =
        reinterpret_cast<const float2 *>(qv) + part * query_run(groups);
    for (int base = 0; base < rows.n; base += kRowsPerPass) {
        const int c = base + quad;
        const bool active = c < rows.n;
        const int row_id = LaneRows::of(rows.id, c), at = LaneRows::of(rows.from, c);
        const float *row = active ? storage + (size_t)row_id * (size_t)d : storage;
        const float s = quad_square_dist_long<CHUNK>(row, qrun, groups, from >> 3,
                                                     part, active);
        if (active && part == 0) dist[at] = s;
    }
}

// Plain rows -> the interleaved layout (row_pair_slot); one thread per pair.
__global__ void interleave_rows(const float *__restrict__ src,
                                float *__restrict__ dst, int64_t n_pairs,
                                int groups) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_pairs) return;
    const int per_row = groups * 4;
    const int64_t r = i / per_row;
    const int p = (int)(i - r * per_row);  // pair p of the row: group p / 4, lane p % 4
    const float2 v = reinterpret_cast<const float2 *>(src)[i];
    *reinterpret_cast<float2 *>(dst + r * (int64_t)groups * 8 +
                                row_pair_slot(p >> 2, p & 3, groups)) = v;
}

// The LDS visited table: 512 buckets of 8 nodes, 8 KB.  A query of the
// headline configuration marks about a thousand nodes: next to no bucket fills
// up, so most queries never touch the bitmask.  Measured per 10 000 queries:
// 1024 x 4 5.76 ms, 2048 x 4 5.77 ms, 1024 x 8 5.52 ms, 512 x 8 5.36 ms.
#ifndef PA_REFINE_SEEN_LOG2
#define PA_REFINE_SEEN_LOG2 9
#endif
#ifndef PA_REFINE_SEEN_WAYS
#define PA_REFINE_SEEN_WAYS 8
#endif
typedef Visited<PA_REFINE_SEEN_LOG2, PA_REFINE_SEEN_WAYS> RefineVisited;

constexpr int kHelped = 4;   // wavefronts of a query when there are few queries
constexpr int kAhead = 8;    // when there are very few
// blocks of a row read at once
template <int WAVES>
constexpr int kRefineChunk = WAVES > 4 ? 4 * PA_LONG_CHUNK
                             : WAVES > 1 ? 2 * PA_LONG_CHUNK : PA_LONG_CHUNK;

#define PA_REFINE_OCCUPANCY(H, WAVES) \
    __attribute__((amdgpu_waves_per_eu((WAVES) > 4 ? 2 : (H) <= 256 || ((WAVES) > 1 && (H) <= 512) ? 4 : (H) <= 384 || ((WAVES) > 1 && (H) <= 1024) ? 3 : (H) <= 1024 ? 2 : 1, 8)))

// WAVES = 1: the wavefront of a query reads its rows itself.  WAVES = 4: three
// more wavefronts wait at a barrier and read rows with it.  A search with the
// device to itself waits for its rows 58 % of the time (768 floats, H = 32):
// 22 rows an expansion are two passes of 16, each of six trips to memory at 8
// blocks a trip; with four wavefronts they are one pass of three trips at 16
// blocks.  Up to H = 512 that is a few registers more than the 128 that four
// wavefronts a SIMD have (12 - 42 spilled).  Measured at H = 32, 768 floats, 1 /
// 512 / 1000 queries: 230 / 393 / 594 us so, 226 / 376 / 774 at three wavefronts a SIMD
// (for which 1000 take two rounds), 248 / 422 / 594 with 8 blocks a trip.  Lists of 2048 cells are held to three wavefronts a SIMD,
// 768 queries at once: 600 / 760 of 768 floats 7.04 / 7.18 ms, where the two that they
// took by themselves leave those batches to one wavefront a query (9.40 / 9.52).
//
// WAVES = 8: seven wavefronts read the rows of nodes the search is about to expand
// (LookAhead), two a node, 32 blocks of a row at a time, and the candidates' rows
// all together.  87 - 92 % of the nodes popped have been asked for, but a node's rows take
// longer than a step, so that what bounds it is still half the waits (4000 of 9500 cycles
// an expansion at one query, H = 32), then the inserts (2400) and the marks (1800).
template <int H, int WAVES>
__global__ __launch_bounds__(kWave *WAVES) PA_REFINE_OCCUPANCY(H, WAVES) void refine_kernel(RefineArgs a) {
    constexpr bool AHEAD = WAVES == kAhead;
    using Ahead = LookAhead<AHEAD ? WAVES - 1 : 0, AHEAD ? 2 : 1>;
    constexpr int kEntries = 0x7fffffff;   // a job: rows of the list in cand_id
    constexpr int S = (H + kWave - 1) / kWave;
    constexpr int kSortN = H <= kWave ? kWave : 1 << (floor_log2(H - 1) + 1);
    constexpr int kHeapCells =
        OpenList<H>::kLdsCells > kSortN ? OpenList<H>::kLdsCells : kSortN;
    struct Lds {
        uint32_t seen_table[RefineVisited::kWords];
        int cand_id[kWave];
        float cand_key[kWave];
        // WAVES > 1: rows to read, from which coordinate; AHEAD: on which graph
        int job_rows, job_from, job_stage;
        int2 heap[kHeapCells];   // open list tail; the sorts reuse it
    };
    __shared__ __align__(16) Lds lds;
    extern __shared__ __align__(16) float qv[];  // the query, query_slot layout
    __shared__ __align__(16) typename Ahead::Slots slots;   // AHEAD
    const int lane = threadIdx.x & (kWave - 1);
    const int d = a.d;
    // A node's row of neighbours, by lane.
    auto neighbours = [&](int stage, int deg, int u) -> int {
        int v = -1;
        if (u < 0) return v;
        if (stage == 0) {
            const int64_t r = a.sub_mapping[u];
            if (r >= 0 && lane < deg) {
                const int w = a.sub_adj[(size_t)r * deg + lane];
                if (w >= 0) v = a.sub_gid[w];
            }
        } else if (lane < deg) {
            v = a.full_adj[(size_t)u * deg + lane];
        }
        return v;
    };
    Ahead ahead{slots, -1, 0, 0};
    if constexpr (AHEAD) {
        const int wave = uni((int)(threadIdx.x / kWave));
        if (threadIdx.x < Ahead::kJobs) Ahead::put(slots.job[threadIdx.x], Ahead::kIdle);
        __syncthreads();   // the only barrier
        if (wave > 0) {
            RefineVisited marks;
            marks.init(lds.seen_table, nullptr, a.n_nodes);
            Ahead::help(slots, lane, [&](int node, int job, int *ids, float *dist) {
                int v, from = 0;
                bool wanted;
                if (node == kEntries) {
                    const int n = Ahead::get(lds.job_rows);
                    from = uni(Ahead::get(lds.job_from));
                    v = lane < n ? lds.cand_id[lane] : -1;
                    wanted = lane < n && lane % (WAVES - 1) == job;
                    dist = lds.cand_key;
                } else {
                    // the part's neighbours, and the distances of those that are
                    // not known to be marked: whatever is new when the node is
                    // popped is among them
                    const int stage = uni(Ahead::get(lds.job_stage));
                    const bool mine = (lane & 1) == job / Ahead::kSlots;
                    v = neighbours(stage, stage == 0 ? a.sub_deg : a.full_deg, node);
                    wanted = Ahead::look_then_show(
                        v, mine, [&](int u) { return marks.known(u); },
                        [] { Ahead::in_order(); }, [&](int u) { Ahead::put(ids[lane], u); });
                }
                eval_lanes_from<kRefineChunk<WAVES>>(a.storage, qv, wanted, v, dist, d, from,
                                                     lane);
            });
            return;
        }
    } else if constexpr (WAVES > 1) {
        // a scalar: the two sides of this branch meet at the same barriers,
        // two per job, and one when the queries are used up
        const int wave = uni((int)(threadIdx.x / kWave));
        if (wave > 0) {
            for (;;) {
                __syncthreads();
                const int n = uni(lds.job_rows);
                if (n < 0) return;
                eval_rows_from<WAVES, kRefineChunk<WAVES>>(a.storage, qv, lds.cand_id,
                                                          lds.cand_key, n, d,
                                                          uni(lds.job_from), lane, wave);
                __syncthreads();
            }
        }
    }
    // distances of the n rows in cand_id over the coordinates [from, d)
    auto eval = [&](int n, int from) {
        if constexpr (AHEAD) {
            lds.job_rows = n, lds.job_from = from;
            ahead.drain(lane);
            ahead.give_all(kEntries, lane);
            ahead.drain(lane);
            Ahead::in_order();
            return;
        }
        if constexpr (WAVES > 1) {
            lds.job_rows = n, lds.job_from = from;
            __syncthreads();
        }
        eval_rows_from<WAVES, kRefineChunk<WAVES>>(a.storage, qv, lds.cand_id,
                                                  lds.cand_key, n, d, from, lane, 0);
        if constexpr (WAVES > 1) __syncthreads();
    };
    float *okey = reinterpret_cast<float *>(lds.heap);
    int *oval = reinterpret_cast<int *>(okey + kHeapCells);
    OpenList<H> open;
    open.cells = lds.heap;
    open.deep = nullptr;  // the whole list in registers and LDS
    int *cand_id = lds.cand_id;
    float *cand_key = lds.cand_key;
    uint32_t *seen = a.seen + (size_t)blockIdx.x * (size_t)a.slot_stride;
    RefineVisited visited;
    visited.init(lds.seen_table, seen, a.n_nodes);
    // The slice is cleared when it is first asked, which most queries never do (a
    // million nodes are 125 KB: one query 170 -> 164 us, 2500 of 768 floats 1321 ->
    // 1287), but in launches of more queries than workgroups at once: 10 000
    // queries 5181 us so, 5266 the other way.  There it is put back to zero after a
    // query that used it; a workgroup's only query leaves it as it is.
    if (a.work_counter) {
        visited.clear(a.words_per_slot, lane);
        visited.zeroed = true;
    }
    for (int turn = 0;;) {
        const int q = next_query(a.work_counter, turn, a.batch, lane);
        if (q >= a.batch) {
            if constexpr (AHEAD) {
                ahead.drain(lane);
                ahead.end(lane);
            } else if constexpr (WAVES > 1) {
                lds.job_rows = -1;
                __syncthreads();
            }
            break;
        }

        unsigned n_expand0 = 0, n_expand1 = 0, n_dist = 0, n_admit = 0, n_tail = 0, n_adj = 0;
#ifdef PA_PHASE_TIMERS
        unsigned long long phase[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#endif
        PA_TIMER_BEGIN();

        if constexpr (AHEAD) ahead.drain(lane);   // of what was asked for in vain
        // empty visited set (it serves both searches), query to LDS
        visited.reset(lane);
        for (int i = lane; i < d; i += kWave)
            qv[query_slot(i, d >> 3)] = a.query[(size_t)q * d + i];
        wave_sync();

        // stage 0: subgraph from the candidates (traverse_cpu.cpp:317-326);
        // stage 1: full graph from the buffer (:327-336)
        for (int stage = 0; stage < 2; ++stage) {
            const int64_t *eI = stage == 0 ? a.init_I + (size_t)q * a.n_init
                                           : a.buf_I + (size_t)q * a.n_buffers;
            float *eD = stage == 0 ? a.init_D + (size_t)q * a.n_init
                                   : a.buf_D + (size_t)q * a.n_buffers;
            const int n_ent = stage == 0 ? a.n_init : a.n_buffers;
            const int tail_from = stage == 0 ? a.dp : d;  // == d: nothing to add
            const int deg = stage == 0 ? a.sub_deg : a.full_deg;
            const int max_iter = stage == 0 ? a.sub_iter : a.full_iter;
            int64_t *oI = stage == 0 ? a.buf_I + (size_t)q * a.n_buffers
                                     : a.out_I + (size_t)q * a.k;
            float *oD = stage == 0 ? a.buf_D + (size_t)q * a.n_buffers
                                   : a.out_D + (size_t)q * a.k;
            const int n_out = stage == 0 ? a.n_buffers : a.k;

            PA_TIMER(0);
            if constexpr (AHEAD) {
                ahead.drain(lane);
                lds.job_stage = stage;
            }
            open.reset(lane);
            // Which node a key of the result list belongs to: beside it in its
            // lane where a lane has one key, else in the log.  Measured with
            // the log for all lists / now, rows of 768 floats: H = 32 one query
            // 251 / 245 us, 1024 612 / 600, 10 000 5.19 / 5.06 ms (5.15 before
            // the log); H = 64 411 / 401, 797 / 759 and 6.31 / 6.18 ms.
            constexpr bool kBeside = S == 1;
            int held = -1;   // kBeside: the node of the lane's key
            ResultKeys<S> res;
            res.init(H, lane);
            ResultLog log;
            log.entry = reinterpret_cast<int2 *>(seen + a.words_per_slot);
            log.capacity = ResultLog::capacity_for(H);
            log.n = 0;
            wave_sync();

            // traverse_cpu.cpp:42-79: complete the entries' distances, mark
            // the entries, push them on the open list in order
            for (int base = 0; base < n_ent; base += kWave) {
                const int i = base + lane;
                int u = -1;
                float dist = INFINITY;
                if (i < n_ent) {
                    const int64_t g = eI[i];
                    dist = eD[i];
                    if (g >= 0 && g < a.n_nodes) u = (int)g;
                }
                if (tail_from < d) {
                    const unsigned long long mask = __ballot(u >= 0);
                    const int n = __popcll(mask);
                    const int rank = lane_rank(mask);
                    if (u >= 0) cand_id[rank] = u;
                    wave_sync();
                    eval(n, tail_from);
                    n_tail += n;
                    wave_sync();
                    PA_TIMER(1);
                    if (u >= 0) {
                        dist += cand_key[rank];
                        eD[i] = dist;
                    }
                    wave_sync();
                }
                visited.mark(u, a.words_per_slot, lane);
                int value = u;
                if constexpr (AHEAD) {
                    if (base == 0) ahead.begin(lane);
                    for (int j = 0; j < 3 && j < max_iter; ++j)
                        ahead.ask_lowest(list_key(dist), value, lane);
                }
                open.push_entries(__ballot(u >= 0), list_key(dist), value, lane);
                PA_TIMER(2);
            }

            // traverse_cpu.cpp:82-136.  The next node's row of neighbour ids is
            // requested before the pop that returns it.  With few queries
            // (WAVES > 1) already when the pop before has shown which node is
            // likely next, and again if an insert put another one first: it
            // is on its way while this node's rows are read.  Where queries
            // fill the device the wasted requests cost more (10 000 queries,
            // 96 floats, H = 96: 2.02 against 1.94 ms).
            constexpr bool kEarly = WAVES > 1;
            auto load_row = [&](int u) -> int { return neighbours(stage, deg, u); };
            // heap_update, traverse_cpu.cpp:25-39, in adjacency order: the lanes'
            // keys and nodes; `value` is what the open list keeps of them
            auto admit = [&](int dk, int id, int value) {
                unsigned long long todo = __ballot(dk < res.worst);
                unsigned long long admitted = 0;
                while (todo) {
                    const int j = __builtin_ctzll(todo);
                    const int dj = __builtin_amdgcn_readlane(dk, j);
                    const int vj = __builtin_amdgcn_readlane(value, j);
                    if (kBeside) {
                        const int node = AHEAD ? __builtin_amdgcn_readlane(id, j) : vj;
                        held = lane == res.holder ? node : held;
                    }
                    open.insert(dj, vj, lane, [&] { res.insert(dj, lane); });
                    admitted |= 1ull << j;
                    todo &= (todo - 1) & __ballot(dk < res.worst);
                }
                if (admitted) {
                    n_admit += __popcll(admitted);
                    if (!kBeside) {
                        log.append(admitted, dk, id, lane);
                        if (log.nearly_full()) log.cut(res.worst, lane);
                    }
                }
            };
            if constexpr (AHEAD) {
                for (int step = 0; step < max_iter; ++step) {
                    const int u = open.root_val();
                    if (u < 0 || open.root_key() >= res.worst) break;
                    typename Ahead::Found found = ahead.find(u & ~Ahead::kAsked, lane);
                    int popped_k, popped_v;
                    open.pop(lane, popped_k, popped_v);
                    n_expand0 += stage == 0, n_expand1 += stage != 0;
                    n_adj += deg;
                    ahead.ids(found, lane);
                    const int v = found.id;
                    if (step + 1 < max_iter) ahead.ask(open.A.v, lane);
                    const bool fresh = visited.mark(v, a.words_per_slot, lane);
                    ahead.take(found, lane);
                    n_dist += __popcll(__ballot(fresh));
                    const int dk = fresh ? list_key(found.dist) : OpenList<H>::kInf;
                    // a neighbour that is before all of the list is next
                    int value = v;
                    if (__ballot(dk < open.root_key()) && ahead.room()) {
                        const int best = ~wave_max_key(~dk);
                        const int at = __builtin_ctzll(__ballot(dk == best));
                        ahead.give(__builtin_amdgcn_readlane(v, at), lane);
                        value = lane == at ? v | Ahead::kAsked : v;
                    }
                    admit(dk, v, value);
                }
            }
            int next = -1, next_row = -1;
            if constexpr (!AHEAD) next = open.root_val(), next_row = load_row(next);
            for (int step = 0; !AHEAD && step < max_iter; ++step) {
                int uk, u;
                open.pop(lane, uk, u);
                PA_TIMER(3);
                if (u < 0 || uk >= res.worst) break;
                n_expand0 += stage == 0, n_expand1 += stage != 0;
                const int v = next_row;
                n_adj += deg;
                const bool fresh = visited.mark(v, a.words_per_slot, lane);
                const unsigned long long mask = __ballot(fresh);
                const int n = __popcll(mask);
                if (kEarly || n == 0) {
                    next = open.root_val();
                    next_row = load_row(next);
                }
                PA_TIMER(4);
                if (n == 0) continue;
                if (fresh) cand_id[lane_rank(mask)] = v;
                wave_sync();
                eval(n, 0);
                n_dist += n;
                wave_sync();
                PA_TIMER(5);
                const int dk = list_key(lane < n ? cand_key[lane] : INFINITY);
                const int id = lane < n ? cand_id[lane] : -1;
                wave_sync();
                admit(dk, id, id);
                const int root = open.root_val();
                if (!kEarly || root != next) next = root, next_row = load_row(root);
                PA_TIMER(6);
            }

            // traverse_cpu.cpp:138-148: now the entries compete for a slot
            wave_sync();
            for (int base = 0; base < n_ent; base += kWave) {
                const int i = base + lane;
                int u = -1;
                float dist = INFINITY;
                if (i < n_ent) {
                    const int64_t g = eI[i];
                    dist = eD[i];
                    if (g >= 0 && g < a.n_nodes) u = (int)g;
                }
                const int dk = list_key(dist);
                unsigned long long todo = __ballot(u >= 0 && dk < res.worst);
                unsigned long long admitted = 0;
                while (todo) {
                    const int j = __builtin_ctzll(todo);
                    todo &= todo - 1;
                    const int dj = __builtin_amdgcn_readlane(dk, j);
                    if (dj >= res.worst) continue;
                    if (kBeside)
                        held = lane == res.holder ? __builtin_amdgcn_readlane(u, j) : held;
                    res.insert(dj, lane);
                    admitted |= 1ull << j;
                }
                if (admitted && !kBeside) {
                    log.append(admitted, dk, u, lane);
                    if (log.nearly_full()) log.cut(res.worst, lane);
                }
            }

            // traverse_cpu.cpp:150-162: best first; with more output slots
            // than heap cells the surplus comes first, as (-1, -inf).  The
            // set is sorted in the LDS the open list no longer needs; from the
            // log it takes every entry below the maximum and of those at it
            // as many as make H.
            wave_sync();
            if (!kBeside) ResultLog::settle();
            for (int i = lane; i < a.sort_n; i += kWave)
                okey[i] = INFINITY, oval[i] = -1;
            wave_sync();
            if (kBeside) {
                if (lane < H) okey[lane] = key_to_float(res.key[0]), oval[lane] = held;
            } else {
                int at_worst = 0;
                for (int base = 0; base < log.n; base += kWave) {
                    const int i = base + lane;
                    at_worst += __popcll(__ballot(i < log.n && log.entry[i].x < res.worst));
                }
                int at_below = 0;
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
                    if (place >= 0 && place < H) okey[place] = key_to_float(e.x), oval[place] = e.y;
                    at_below += __popcll(mb);
                    at_worst += __popcll(mt);
                }
            }
            wave_sync();
            for (int size = 2; size <= a.sort_n; size <<= 1) {
                for (int stride = size >> 1; stride > 0; stride >>= 1) {
                    for (int t = lane; t < (a.sort_n >> 1); t += kWave) {
                        const int i = ((t & ~(stride - 1)) << 1) | (t & (stride - 1));
                        const int j = i | stride;
                        const float ki = okey[i], kj = okey[j];
                        const int vi = oval[i], vj = oval[j];
                        const bool gt = ki > kj || (ki == kj && vi > vj);
                        const bool lt = ki < kj || (ki == kj && vi < vj);
                        if ((i & size) == 0 ? gt : lt) {
                            okey[i] = kj, oval[i] = vj;
                            okey[j] = ki, oval[j] = vi;
                        }
                    }
                    wave_sync();
                }
            }
            const int surplus = n_out > H ? n_out - H : 0;
            for (int i = lane; i < n_out; i += kWave) {
                const int e = i - surplus;
                oI[i] = e < 0 ? (int64_t)-1 : (int64_t)oval[e];
                oD[i] = e < 0 ? -INFINITY : okey[e];
            }
            // the buffer is read back as the next search's entries, by other
            // lanes than those that wrote it
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            wave_sync();
            PA_TIMER(7);
        }

        if (a.work_counter) visited.clean(a.words_per_slot, lane);

        if (a.counters && lane == 0) {
            atomicAdd(&a.counters[0], (unsigned long long)n_expand0);
            atomicAdd(&a.counters[1], (unsigned long long)n_expand1);
            atomicAdd(&a.counters[2], (unsigned long long)n_dist);
            atomicAdd(&a.counters[3], (unsigned long long)n_admit);
            atomicAdd(&a.counters[4], (unsigned long long)n_tail);
            atomicAdd(&a.counters[5], (unsigned long long)n_adj);
#ifdef PA_PHASE_TIMERS
            for (int i = 0; i < 8; ++i) atomicAdd(&a.counters[6 + i], phase[i]);
#endif
        }
    }
}

typedef void (*RefineFn)(RefineArgs);

template <int WAVES>
RefineFn pick_kernel(int H) {
    switch (H) {
        case 16: return refine_kernel<16, WAVES>;
        case 32: return refine_kernel<32, WAVES>;
        case 48: return refine_kernel<48, WAVES>;
        case 64: return refine_kernel<64, WAVES>;
        case 96: return refine_kernel<96, WAVES>;
        case 128: return refine_kernel<128, WAVES>;
        case 192: return refine_kernel<192, WAVES>;
        case 256: return refine_kernel<256, WAVES>;
        case 384: return refine_kernel<384, WAVES>;
        case 512: return refine_kernel<512, WAVES>;
        case 1024: return refine_kernel<1024, WAVES>;
        case 2048: return refine_kernel<2048, WAVES>;
        default: return nullptr;
    }
}

int round_up(int64_t x, int64_t m) { return (int)(((x + m - 1) / m) * m); }

struct Plan {
    int H, sort_n, lds_bytes, n_slots, words_per_slot, slot_stride, threads;
    size_t workspace_bytes;
    RefineFn fn;
};

#ifndef PA_REFINE_MAX_WAVES
#define PA_REFINE_MAX_WAVES 20
#endif
constexpr int kMaxWavesPerCu = PA_REFINE_MAX_WAVES;

// Workgroups of `fn` the current device holds at once (none where one does not fit a
// compute unit's LDS).
int residency(RefineFn fn, int threads, int lds_bytes, int *slots) {
    int dev = 0, cus = 0, per_cu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    // the residency of a (device, kernel, LDS size) never changes
    static std::mutex mutex;
    static std::map<std::tuple<int, const void *, int>, int> known;
    std::lock_guard<std::mutex> guard(mutex);
    const auto key = std::make_tuple(dev, reinterpret_cast<const void *>(fn), lds_bytes);
    auto it = known.find(key);
    if (it == known.end()) {
        e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e == hipSuccess)
            e = workgroups_per_cu(reinterpret_cast<const void *>(fn), dev, threads, lds_bytes,
                                  &per_cu);
        if (e != hipSuccess) return (int)e;
        if (per_cu > kMaxWavesPerCu) per_cu = kMaxWavesPerCu;
        it = known.emplace(key, per_cu * cus).first;
    }
    *slots = it->second;
    return PA_OK;
}

// `beside`: queries of other launches at the same time.  It decides about the
// form alone: one wavefront per query never takes more slots than four.
int make_plan(int64_t n_nodes, int64_t batch, int64_t beside, int d, int ef_search, Plan *p) {
    if (n_nodes <= 0 || batch < 0 || beside < 0) return PA_E_SHAPE;
    if (n_nodes >= (1ll << 31)) return PA_E_RANGE;
    if (d <= 0 || d % 8) return PA_E_DIM;
    if (ef_search < 1 || ef_search > PA_MAX_EF_TOTAL) return PA_E_EF;
    p->H = pa_heap_size(ef_search);
    p->sort_n = kWave;
    while (p->sort_n < p->H) p->sort_n <<= 1;
    p->lds_bytes = query_floats(d) * 4;
    // Four wavefronts per query as long as every query, those of launches beside
    // this one too, has its workgroup at once (1024 queries at H <= 512).  Measured on
    // 1M x 768, one / four, us: H = 32, one query 342 / 230 (the median of 60), 37 431 / 263,
    // 512 587 / 393; H = 512, 1000 3574 / 2949; beyond that the wavefronts that only read rows
    // take the place of queries: H = 32, 1500 854 / 990, H = 512 3860 / 5216; 96 floats, H = 64
    // 419 / 678; two launches of 1250 at a time, H = 128, 2976 / 3604 (of 1000, which would
    // be two full rounds, 2747 / 2205).
    // Eight where a compute unit has one query at most, seven of them helpers that
    // read ahead.  Four / eight: H = 32, 768 floats, one query 230 / 182, 37 263 / 218, 256
    // 320 / 283; H = 128, 37 621 / 490; H = 512, 37 1981 / 1908; 96 floats, H = 64, 256 299 /
    // 265.  With half the registers and two queries a compute unit, rows in three trips
    // instead of two, they were at 204 us for one query of H = 32 and 512 at 491 against 466.
    // (Their slots are 4 KB of LDS: of the longest rows a query fits beside them in the
    // other forms alone, and has no workgroup here.)
    p->threads = kAhead * kWave;
    p->fn = pick_kernel<kAhead>(p->H);
    if (!p->fn) return PA_E_EF;
    int slots = 0;
    int rc = residency(p->fn, p->threads, p->lds_bytes, &slots);
    if (rc != PA_OK) return rc;
    if (batch > slots - beside || n_nodes >= LookAhead<1>::kAsked) {
        p->threads = kHelped * kWave;
        p->fn = pick_kernel<kHelped>(p->H);
        rc = residency(p->fn, p->threads, p->lds_bytes, &slots);
        if (rc != PA_OK) return rc;
    }
    if (batch > slots - beside) {
        p->threads = kWave;
        p->fn = pick_kernel<1>(p->H);
        rc = residency(p->fn, p->threads, p->lds_bytes, &slots);
        if (rc != PA_OK) return rc;
    }
    if (slots > batch) slots = (int)batch;
    if (slots < 1) slots = 1;   // (no query, or rows that fit no form: the launch says so)
    p->n_slots = slots;
    p->words_per_slot = round_up((n_nodes + 31) / 32, kSlotAlignWords);
    // a slot: the visited slice, then the log of admitted candidates (lists of
    // more than one key a lane)
    p->slot_stride =
        p->words_per_slot + (p->H > kWave ? 2 * ResultLog::capacity_for(p->H) : 0);
    p->workspace_bytes =
        kWorkCounterBytes + (size_t)p->n_slots * p->slot_stride * 4;
    return PA_OK;
}

}  // namespace

extern "C" int pa_rows_prepare(float *dst, const float *src, int64_t n_rows,
                               int d_model, void *stream_) {
    if (n_rows < 0) return PA_E_SHAPE;
    if (d_model <= 0 || d_model % 8) return PA_E_DIM;
    if (n_rows == 0) return PA_OK;
    if (!dst || !src || dst == src) return PA_E_NULL;
    const int64_t n_pairs = n_rows * (d_model / 2);
    if ((n_pairs + 255) / 256 >= (1ll << 31)) return PA_E_RANGE;
    interleave_rows<<<(unsigned)((n_pairs + 255) / 256), 256, 0,
                      (hipStream_t)stream_>>>(src, dst, n_pairs, d_model / 8);
    return (int)hipGetLastError();
}

extern "C" int pa_refine_plan(int64_t n_nodes, int64_t batch, int d_model,
                              int ef_search, int *n_slots,
                              size_t *workspace_bytes) {
    Plan p;
    const int rc = make_plan(n_nodes, batch, 0, d_model, ef_search, &p);
    if (rc != PA_OK) return rc;
    if (n_slots) *n_slots = p.n_slots;
    if (workspace_bytes) *workspace_bytes = p.workspace_bytes;
    return PA_OK;
}

extern "C" int pa_refine_form(int64_t n_nodes, int64_t batch, int64_t beside, int d_model,
                              int ef_search, int *wavefronts) {
    Plan p;
    const int rc = make_plan(n_nodes, batch, beside, d_model, ef_search, &p);
    if (rc != PA_OK) return rc;
    if (wavefronts) *wavefronts = p.threads == kWave ? 1 : kHelped;
    return PA_OK;
}

extern "C" int pa_refine_wavefronts(int64_t n_nodes, int64_t batch, int64_t beside,
                                    int d_model, int ef_search, int *wavefronts) {
    Plan p;
    const int rc = make_plan(n_nodes, batch, beside, d_model, ef_search, &p);
    if (rc != PA_OK) return rc;
    if (wavefronts) *wavefronts = p.threads / kWave;
    return PA_OK;
}

extern "C" int pa_refine_beside(int64_t *out_I, float *out_D, int64_t *buf_I, float *buf_D,
                                const int64_t *init_I, float *init_D, const int32_t *sub_adj,
                                const int32_t *sub_gid, const int64_t *sub_mapping,
                                const int32_t *full_adj, const float *storage,
                                const float *query, int64_t batch, int64_t beside,
                                int64_t n_nodes, int d_model, int d_principle, int n_init,
                                int n_buffers, int k, int ef_search, int sub_neighbors,
                                int full_neighbors, void *workspace, size_t workspace_bytes,
                                uint64_t *counters, void *stream_) {
    if (batch < 0 || n_nodes <= 0 || n_init < 0 || n_buffers < 0 || k < 0)
        return PA_E_SHAPE;
    if (n_nodes >= (1ll << 31) || batch >= (1ll << 31)) return PA_E_RANGE;
    if (sub_neighbors < 1 || sub_neighbors > PA_MAX_NEIGHBORS ||
        full_neighbors < 1 || full_neighbors > PA_MAX_NEIGHBORS)
        return PA_E_NEIGHBORS;
    if (d_principle <= 0 || d_principle > d_model || d_principle % 8)
        return PA_E_DIM;
    Plan p;
    const int rc = make_plan(n_nodes, batch, beside, d_model, ef_search, &p);
    if (rc != PA_OK) return rc;
    if (batch == 0) return PA_OK;
    if (!out_I || !out_D || !buf_I || !buf_D || !sub_adj || !sub_gid ||
        !sub_mapping || !full_adj || !storage || !query || !workspace ||
        (n_init > 0 && (!init_I || !init_D)))
        return PA_E_NULL;
    if (workspace_bytes < p.workspace_bytes) return PA_E_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(workspace) % 256) return PA_E_WORKSPACE;

    RefineArgs a;
    a.out_I = out_I, a.out_D = out_D, a.buf_I = buf_I, a.buf_D = buf_D;
    a.init_I = init_I, a.init_D = init_D;
    a.sub_adj = sub_adj, a.sub_gid = sub_gid, a.sub_mapping = sub_mapping;
    a.full_adj = full_adj, a.storage = storage, a.query = query;
    a.work_counter = p.n_slots < batch ? reinterpret_cast<int *>(workspace) : nullptr;
    a.seen = reinterpret_cast<uint32_t *>(
        reinterpret_cast<unsigned char *>(workspace) + kWorkCounterBytes);
    a.counters = reinterpret_cast<unsigned long long *>(counters);
    a.batch = (int)batch, a.n_nodes = (int)n_nodes;
    a.d = d_model, a.dp = d_principle;
    a.n_init = n_init, a.n_buffers = n_buffers, a.k = k, a.H = p.H;
    a.sub_deg = sub_neighbors, a.full_deg = full_neighbors;
    // traverse_cpu.cpp:82 with the limits of :325 (REFINE_STEP) and :18 (1024)
    a.sub_iter = 2 * ef_search < 2 ? 2 * ef_search : 2;
    a.full_iter = 2 * ef_search < 1024 ? 2 * ef_search : 1024;
    a.words_per_slot = p.words_per_slot, a.slot_stride = p.slot_stride;
    a.sort_n = p.sort_n;

    hipStream_t stream = (hipStream_t)stream_;
    if (a.work_counter) reset_refine_counter<<<1, 1, 0, stream>>>(a.work_counter);
    p.fn<<<p.n_slots, p.threads, p.lds_bytes, stream>>>(a);
    return (int)hipGetLastError();
}

extern "C" int pa_refine(int64_t *out_I, float *out_D, int64_t *buf_I,
                         float *buf_D, const int64_t *init_I, float *init_D,
                         const int32_t *sub_adj, const int32_t *sub_gid,
                         const int64_t *sub_mapping, const int32_t *full_adj,
                         const float *storage, const float *query,
                         int64_t batch, int64_t n_nodes, int d_model,
                         int d_principle, int n_init, int n_buffers, int k,
                         int ef_search, int sub_neighbors, int full_neighbors,
                         void *workspace, size_t workspace_bytes,
                         uint64_t *counters, void *stream_) {
    return pa_refine_beside(out_I, out_D, buf_I, buf_D, init_I, init_D, sub_adj, sub_gid,
                            sub_mapping, full_adj, storage, query, batch, 0, n_nodes,
                            d_model, d_principle, n_init, n_buffers, k, ef_search,
                            sub_neighbors, full_neighbors, workspace, workspace_bytes,
                            counters, stream_);
}
