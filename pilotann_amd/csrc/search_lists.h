// Device-side lists of the per-query search, shared by the subgraph traversal
// and the full-dimension refine (gfx950, one 64-lane wavefront per query): the
// open list (the reference's array heap, extension/inc/heapq.cuh:13-88, top
// levels in registers), the result list, the exact visited table of the refine,
// and the batched row distances.
#ifndef PILOTANN_SEARCH_LISTS_H
#define PILOTANN_SEARCH_LISTS_H

#include "device_common.h"

namespace pa {

constexpr int kSlotAlignWords = 256;   // bitmask slice: multiple of 1 KiB
constexpr int kWorkCounterBytes = 256; // head of the workspace
#ifndef PA_SEEN_LOG2
#define PA_SEEN_LOG2 10
#endif
constexpr int kSeenCacheLog2 = PA_SEEN_LOG2;
constexpr int kSeenCache = 1 << kSeenCacheLog2;  // LDS words remembering visited rows

// The next query of a workgroup.  Where every query has its workgroup (no
// `counter`) it is the workgroup's own number, once: no launch that sets a
// counter, no trip to memory for it.  `turn`: how many this workgroup had.
__device__ __forceinline__ int next_query(int *counter, int &turn, int batch, int lane) {
    if (!counter) return turn++ ? batch : (int)blockIdx.x;
    int q = 0;
    if (lane == 0) q = atomicAdd(counter, 1);
    return uni(q);
}

// ---- open list: heapq.cuh, top of the heap in registers ----------------------
//
// The reference's open list is an array heap of 2H cells with the sift rules
// of extension/inc/heapq.cuh:13-88.  Here node i of that array is node
// j = i + 1 (children 2j and 2j + 1), level L holds j in [2^L, 2^(L+1)).
//
// Levels 0..8 live in registers.  Bank A holds levels 0..5, node j in lane j;
// below that every lane has a subtree of its own: node 64 + lane (bank B), its
// children (C and D), its grandchildren (E F under C, G I under D) and, in a
// list of 512 cells, the one node of level 9 (J, lane 0).  Longer lists have
// the levels from 9 on in LDS at [j - 512] as (key, value), a sibling pair per
// aligned 16 bytes; with DEEP the levels from DEEP on sit in device memory
// instead (the wavefront's own region, at [j - 2^DEEP], same cells): a long
// list then takes less LDS, more wavefronts fit a compute unit, and a walk pays
// one memory round trip per such level.  Keys are kept as order-preserving
// integers (float_to_key).  After each operation the heap is, cell for cell,
// the reference's.
//
// In the registers nothing is walked.  Which child of every node a path takes
// is decided for all nodes at once (one comparison with the sibling), a node is
// on the path if everything above it is taken too (one lane mask and two
// vector instructions), and every node on the path takes its parent's or its
// child's entry in the same instructions.  What bounds it is the chain of
// dependent instructions: a vector one takes a wavefront 4 cycles, a scalar one
// 8, a lane gather or an LDS read 50 - 60, a value that crosses from one unit to the
// other 12 - 20.  Measured, one wavefront, cycles for a pop / for an insert with
// the result list's, against paths walked on the scalar unit (three instructions
// a level) with levels 8 and on in LDS: lists of 64 cells 416 / 537 -> 204 / 288,
// of 256 584 / 602 -> 236 / 332, of 512 695 / 669 -> 296 / 388, of 2048 860 / 911 ->
// 541 / 745.  In the searches: 100 000 rows of 32 floats, H = 256, 128 queries 495
// -> 405 us; a million rows, 250 000 of 128 floats, H = 128, one query 334 -> 262
// us (the median of 60); 10 000 queries, rows of 64 floats, H = 256 2.60 -> 2.26 ms; H = 1024,
// 500 000 rows of 128 floats 19.7 -> 17.7 ms.
__device__ __forceinline__ int float_to_key(float x) {
    const int b = __float_as_int(x);
    return b ^ ((b >> 31) & 0x7fffffff);
}
// The key an entry has in the lists: above 0x80000000, which stands for "below
// every key".  (That is the image of one NaN, which so counts as the key after.)
__device__ __forceinline__ int list_key(float x) {
    return max(float_to_key(x), (int)0x80000001);
}
__device__ __forceinline__ float key_to_float(int k) {
    return __int_as_float(k ^ ((k >> 31) & 0x7fffffff));
}

__device__ __forceinline__ int med3(int a, int b, int c) {
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

constexpr int floor_log2(int x) { return x <= 1 ? 0 : 1 + floor_log2(x >> 1); }

// Cells of an open list of 2H cells that sit in device memory when the levels
// from `deep` on do (0: none do).
constexpr int open_list_deep_cells(int H, int deep) {
    return deep >= 10 && deep < floor_log2(2 * H) ? 2 * H - (1 << deep) : 0;
}

template <int H, int DEEP = 0>
struct OpenList {
    static constexpr int kSize = 2 * H;           // cells of the reference heap
    static constexpr int kDepth = floor_log2(kSize);  // deepest level
    static constexpr int kRegNodes = 512;
    static constexpr bool kLong = kSize > kRegNodes;  // levels 9 and on in LDS
    // the deepest level has one node (J), or, in a list of 768 cells, every other
    static constexpr bool kOneLast = kSize == 1 << kDepth;
    static constexpr int kEnd = kOneLast ? kDepth - 1 : kDepth;  // last level below J
    static constexpr int kDeepCells = open_list_deep_cells(H, DEEP);
    static constexpr int kDeepFrom = kDeepCells ? DEEP : kDepth + 1;
    static constexpr int kDeepBase = 1 << kDeepFrom;  // first node in device memory
    // (the pair after the last one is for the lanes off a path)
    static constexpr int kNowhere = kDeepCells ? kDeepBase : kOneLast ? kSize : kSize + 2;
    static constexpr int kLdsCells = !kLong ? 0 : kNowhere + 2 - kRegNodes;
    // The last level of the shorter lists is not complete: the lane that has its
    // last node, a left child without a sibling.
    static constexpr int kLast = kDepth == 5   ? kSize
                                 : kDepth == 6 ? kSize - 64
                                 : kDepth == 7 ? (kSize - 128) / 2
                                 : kDepth == 8 ? (kSize - 256) / 4
                                               : kWave;
    static constexpr int kInf = 0x7f800000;       // float_to_key(+inf)
    static constexpr int kBelowAll = (int)0x80000000;
    static constexpr int kAboveAll = 0x7fffffff;

    struct Cell {
        int k, v;
    };
    Cell A, B, C, D, E, F, G, I, J;
    int2 *cells;  // node j in [512, kDeepBase) at [j - 512] as (key, value); 16-byte aligned
    int2 *deep;   // node j >= kDeepBase at [j - kDeepBase], device memory, 16-byte aligned
    // Lane constants (reset()).  The lanes of bank A with the nodes from level 1
    // down to this lane's node of bank A, and down to the parent of its node of
    // bank B.
    int wayA_lo, wayA_hi, wayB_lo, wayB_hi;
    int left;             // 1 in a pair's left lane, else 0
    int tieA, tieB;       // see path()
    int4 pending;   // pop(): the requested pair of level kDeepFrom, until pop_finish()
    int pending_j;  // its parent, 0: nothing pending

    __device__ __forceinline__ static int rl(int x, int l) {
        return __builtin_amdgcn_readlane(x, l);
    }
    __device__ __forceinline__ int root_key() const { return rl(A.k, 1); }
    __device__ __forceinline__ int root_val() const { return rl(A.v, 1); }
    // the entry of another lane of a bank, taken modulo 64, by the lane's number
    // times four
    __device__ __forceinline__ static Cell of_lane(const Cell &bank, int l4) {
        return {__builtin_amdgcn_ds_bpermute(l4, bank.k),
                __builtin_amdgcn_ds_bpermute(l4, bank.v)};
    }
    // x, made anew where it is used: one instruction instead of a register that
    // is held through the whole search
    __device__ __forceinline__ static int here(int x) {
        asm volatile("" : "+v"(x));
        return x;
    }
    __device__ __forceinline__ static Cell pick(bool first, const Cell &a, const Cell &b) {
        return {first ? a.k : b.k, first ? a.v : b.v};
    }
    __device__ __forceinline__ static Cell none() { return {kInf, -1}; }

    static constexpr int kToBelowAll = (int)0xff800000;  // kInf less this: kBelowAll
    static constexpr int kNoWay = 0xc;   // both children of the root: no path has them
    // For bank A, level 1 and down: the lanes of node j and of what is above it
    // (lane 0, which holds no node: no way).
    __device__ __forceinline__ static unsigned long long way_to(int j) {
        unsigned long long way = j == 0 ? kNoWay : 0;
        for (; j > 1; j >>= 1) way |= 1ull << j;
        return way;
    }

    __device__ __forceinline__ void reset(int lane) {
        const unsigned long long way = way_to(lane), way5 = way_to(32 + (lane >> 1));
        wayA_lo = (int)way, wayA_hi = (int)(way >> 32);
        wayB_lo = (int)way5, wayB_hi = (int)(way5 >> 32);
        left = 1 & ~lane;
        tieA = tieB = left;
        if (kDepth == 5 && lane == kLast) tieA = kToBelowAll;
        if (kDepth == 5 && lane > kLast) wayA_lo = kNoWay;
        if (kDepth == 6 && lane == kLast) tieB = kToBelowAll;
        if (kDepth == 6 && lane > kLast) wayB_lo = kNoWay;
        A = B = C = D = E = F = G = I = J = none();
        if (lane == 0) A.k = kBelowAll;  // lane 0 of bank A holds no node: the root's parent
        for (int i = lane; i < kLdsCells; i += kWave) cells[i] = make_int2(kInf, -1);
        for (int i = lane; i < kDeepCells; i += kWave) deep[i] = make_int2(kInf, -1);
        pending_j = 0;
    }

    // The path from the root that takes the larger child (left on ties) or the
    // smaller one (left on ties), for all lanes at once and without walking it.
    // Of a pair's two in banks A and B, the left one is taken if it is not below
    // (above) the right one, which is one integer away from "above (below)"
    // (`left`).  Cells that the reference's heap does not have hold (inf, -1).  A
    // pop's path may run on into them; the large leaf's must not: in banks A
    // and B their lanes have no way, and a node without a sibling is taken because
    // its tie constant makes the sibling's infinity smaller than every key
    // (further down: on()).
    struct Path {
        int offA, offB;     // 0: all above and, in bank A, the lane's node are taken
        bool takenB;        // the lane's node of bank B is taken
        bool right, rightC, rightD;   // of the children of B, C, D the right one is
    };
    __device__ __forceinline__ static int less(int a, int b) {   // modulo 2^32
        return (int)((unsigned)a - (unsigned)b);
    }
    template <bool LARGER>
    __device__ __forceinline__ Path path() const {
        Path w;
        const int sa = __builtin_amdgcn_mov_dpp(A.k, 0xB1, 0xF, 0xF, true);
        const unsigned long long not_taken =
            __ballot(LARGER ? A.k <= less(sa, tieA) : A.k >= sa + left);
        const int lo = (int)not_taken, hi = (int)(not_taken >> 32);
        w.offB = 0, w.takenB = w.right = w.rightC = w.rightD = false;
        if (kDepth >= 6) {
            const int sb = __builtin_amdgcn_mov_dpp(B.k, 0xB1, 0xF, 0xF, true);
            w.takenB = LARGER ? B.k > less(sb, tieB) : B.k < sb + left;
        }
        if (kDepth >= 7) w.right = LARGER ? D.k > C.k : D.k < C.k;
        if (kDepth >= 8 && kLast > 0) {
            w.rightC = LARGER ? F.k > E.k : F.k < E.k;
            w.rightD = LARGER ? I.k > G.k : I.k < G.k;
        }
        w.offA = (hi & wayA_hi) | (lo & wayA_lo);
        if (kDepth >= 6) w.offB = (hi & wayB_hi) | (lo & wayB_lo);
        return w;
    }
    // `yes` for the cells on a path, `no` for the others.
    struct Spread {
        int A, B, C, D, E, F, G, I, J;
    };
    template <bool LARGER>
    __device__ __forceinline__ static Spread on(const Path &w, int yes, int no, int lane) {
        Spread t;
        t.A = w.offA == 0 ? yes : no;
        const int taken = w.takenB ? yes : no;
        t.B = w.offB == 0 ? taken : no;
        t.C = w.right ? no : t.B, t.D = w.right ? t.B : no;
        if (LARGER && kDepth == 7) {
            t.C = lane == kLast ? t.B : lane > kLast ? no : t.C;
            t.D = lane >= kLast ? no : t.D;
        }
        if (kDepth == 8 && kLast == 0) {
            t.E = lane == 0 ? t.C : no;
            t.F = t.G = t.I = no;
        } else {
            int c = t.C, d = t.D;
            bool rightC = w.rightC;
            if (LARGER && kDepth == 8) {
                c = lane <= kLast ? c : no, d = lane < kLast ? d : no;
                rightC = rightC && lane != kLast;
            }
            t.E = rightC ? no : c, t.F = rightC ? c : no;
            t.G = w.rightD ? no : d, t.I = w.rightD ? d : no;
        }
        t.J = lane == 0 ? t.E : no;
        return t;
    }
    // Long lists: the lane's node on level 8 that a path through its subtree
    // takes, and its entry.
    __device__ __forceinline__ static int node8(const Path &w, int lane) {
        const int under_d = w.rightD ? 3 : 2, under_c = w.rightC ? 1 : 0;
        return 256 + 4 * lane + (w.right ? under_d : under_c);
    }
    __device__ __forceinline__ Cell at8(const Path &w) const {
        return pick(w.right, pick(w.rightD, I, G), pick(w.rightC, F, E));
    }

    // ---- levels below the registers: 3 LDS, 4 device memory.  A cell is only ever
    // read and written by the lane that has the subtree it is in; lanes off a path
    // read and write the pair kNowhere in LDS and nothing in device memory.

    __device__ __forceinline__ static constexpr int kind(int level) {
        return level < kDeepFrom ? 3 : 4;
    }
    // the sibling pair (c, c + 1), c even: one 16-byte read
    __device__ __forceinline__ int4 pair(const int KIND, int c, bool on) const {
        if (KIND == 3)
            return *reinterpret_cast<const int4 *>(cells + ((on ? c : kNowhere) - kRegNodes));
        int4 p = make_int4(kInf, -1, kInf, -1);
        if (on) p = *reinterpret_cast<const int4 *>(deep + (c - kDeepBase));
        return p;
    }
    __device__ __forceinline__ void put(const int KIND, int j, int k, int v, bool on) {
        if (KIND == 3) cells[(on ? j : kNowhere) - kRegNodes] = make_int2(k, v);
        else if (on) deep[j - kDeepBase] = make_int2(k, v);
    }

    // ---- pop

    // The smaller of every sibling pair of a bank (left on ties), in the left
    // lane of the pair.
    __device__ __forceinline__ static Cell smaller_of_pair(const Cell &c) {
        const Cell s = {__builtin_amdgcn_mov_dpp(c.k, 0xB1, 0xF, 0xF, true),
                        __builtin_amdgcn_mov_dpp(c.v, 0xB1, 0xF, 0xF, true)};
        return {min(c.k, s.k), s.k < c.k ? s.v : c.v};
    }
    // heapq.cuh:37-45 with the sift of :13-29: the root leaves, (inf, -1)
    // sinks along the smaller child (left on ties).  The reference stops when
    // that child is (inf, -1) too; going on to the bottom instead only copies
    // (inf, -1) over (inf, -1) — every infinite cell carries -1 — so the
    // final state is the same.  Every node on the path takes the entry of its
    // smaller child, the last one (inf, -1): the smaller children of bank A are
    // a lane gather away (of bank A, of bank B for level 5), the others in the
    // lane itself.
    __device__ __forceinline__ void pop(int lane, int &out_k, int &out_v) {
        out_k = root_key();
        out_v = root_val();
        const int left4 = here(lane) << 3;   // the left child's lane
        const Cell underA = of_lane(smaller_of_pair(A), left4);
        const Cell under5 = kDepth >= 6 ? of_lane(smaller_of_pair(B), left4) : none();
        __builtin_amdgcn_sched_barrier(0);   // they travel while the path is found
        const Path w = path<false>();
        Cell under8 = none();
        // long lists: the node on level 9 that is to be filled, and whether this
        // lane has it
        int j = 0;
        bool mine = false;
        if (kLong) {
            j = 2 * node8(w, lane);
            mine = w.takenB && w.offB == 0;
            if (kDepth == 9) mine = mine && j <= kSize;
            const int4 p = pair(kind(9), j, mine);
            // node kSize has no sibling
            const bool right = p.z < p.x && !(kDepth == 9 && j == kSize);
            under8 = {right ? p.z : p.x, right ? p.w : p.y};
            if (kDepth == 9) under8 = pick(mine, under8, none());
            j += right;
        }
        const Spread t = on<false>(w, 0, 1, lane);
        const Cell underB = kDepth >= 7 ? pick(w.right, D, C) : none();
        const Cell underC = kDepth >= 8 ? pick(w.rightC, F, E) : none();
        const Cell underD = kDepth >= 8 && kLast > 0 ? pick(w.rightD, I, G) : none();
        A = pick(t.A == 0, pick(lane >= 32, under5, underA), A);
        if (kDepth >= 6) B = pick(t.B == 0, underB, B);
        if (kDepth >= 7) C = pick(t.C == 0, underC, C), D = pick(t.D == 0, underD, D);
        if (kDepth >= 8) E = pick(t.E == 0, kSize == 512 ? J : under8, E);
        if (kDepth >= 8 && kLast > 0) {
            F = pick(t.F == 0, under8, F);
            G = pick(t.G == 0, under8, G);
            I = pick(t.I == 0, under8, I);
        }
        if (kSize == 512) J = pick(t.J == 0, none(), J);
        pending_j = 0;
        if (kLong) pop_below(j, mine, false);
    }
    // The levels from 10 on: cell j, on level 9, has given its entry away.  With
    // levels in device memory pop() only requests the first pair it needs from
    // there; the caller puts the work that does not touch the list (the root is
    // in registers) between pop() and pop_finish(), which comes before the next
    // insert or pop.
    __device__ __forceinline__ void pop_below(int j, bool mine, const bool FINISH) {
#pragma unroll
        for (int L = FINISH ? kDeepFrom : 10; L <= kEnd; ++L) {
            int4 p;
            if (kDeepCells && L == kDeepFrom) {
                if (!FINISH) {
                    pending = pair(4, 2 * j, mine);
                    pending_j = mine ? j : 0;
                    return;
                }
                p = pending;
            } else {
                p = pair(kind(L), 2 * j, mine);
            }
            const bool right = p.z < p.x;
            put(kind(L - 1), j, right ? p.z : p.x, right ? p.w : p.y, mine);
            j = 2 * j + right;
        }
        const bool above = kOneLast && 2 * j == kSize;   // (a node of lane 0's)
        put(kind(kEnd), j, above ? J.k : kInf, above ? J.v : -1, mine);
        if (kOneLast) J = pick(above && mine, none(), J);
    }
    __device__ __forceinline__ void pop_finish() {
        if (!kDeepCells || !__ballot(pending_j != 0)) return;
        const int j = pending_j;
        pending_j = 0;
        pop_below(j, j != 0, true);
    }

    // ---- insert
    //
    // heapq.cuh:47-77: walk to a leaf through the larger child (left on
    // ties), overwrite it when the new key is strictly smaller, let the new
    // entry rise: along the path, whose keys do not fall from the root down,
    // every entry with a larger key moves one level down and the new one takes
    // the place of the highest of them.  A new key that is not below the leaf's
    // is not below any key of the path, and nothing moves.

    // The parents' entries of bank A's and bank B's nodes.
    struct Parents {
        Cell A, B;
    };
    __device__ __forceinline__ Parents parents(int lane) const {
        Parents up;
        const int above4 = here(lane) << 1;   // (bits 0 and 1 don't count)
        up.A = of_lane(A, above4);
        up.B = kDepth >= 6 ? of_lane(A, above4 + 128) : none();
        return up;
    }
    // The registers.  A node on the path takes the median of its parent's key,
    // its own and the new one, and the value that goes with that; a node off the
    // path does the same with the largest key for the new one, which changes
    // nothing (a parent's key is never above its child's).
    __device__ __forceinline__ static bool take(Cell &c, const Cell &up, int key, int moved) {
        const bool moves = c.k > key;
        c.k = med3(up.k, key, c.k);
        c.v = moves ? moved : c.v;
        return moves;
    }
    // Returns whether the lane has a node that took another entry.
    __device__ __forceinline__ bool shift(const Path &w, const Parents &up, int k, int v,
                                          int lane) {
        const Spread t = on<true>(w, k, kAboveAll, lane);
        // what a node that changes takes: its parent's value or the new one
        const int toA = up.A.k > k ? up.A.v : v, toB = up.B.k > k ? up.B.v : v;
        const int toC = B.k > k ? B.v : v;
        bool any = false;
        if (kDepth >= 8) {
            const int toE = C.k > k ? C.v : v;
            if (kSize == 512) any |= take(J, E, t.J, E.k > k ? E.v : v);
            any |= take(E, C, t.E, toE);
            if (kLast > 0) {
                const int toG = D.k > k ? D.v : v;
                any |= take(F, C, t.F, toE);
                any |= take(G, D, t.G, toG);
                any |= take(I, D, t.I, toG);
            }
        }
        if (kDepth >= 7) any |= take(C, B, t.C, toC), any |= take(D, B, t.D, toC);
        if (kDepth >= 6) any |= take(B, up.B, t.B, toB);
        any |= take(A, up.A, t.A, toA);
        return any;
    }

    // Long lists: the path below level 8, in the lane whose subtree it is in.
    struct Low {
        bool mine;
        int j;        // the path's node on level kEnd
        bool bottom;  // list of 768 cells: it has one there
        static constexpr int kLow = kLong ? kEnd - 7 : 1;
        Cell at[kLow];   // its entries of levels 8 .. kEnd
    };
    // `beside` is work of the caller's that does not touch the list, placed where
    // the first pair travels.
    template <class WORK>
    __device__ __forceinline__ Low walk(const Path &w, int lane, const WORK &beside) const {
        Low low;
        int j = node8(w, lane);
        low.mine = w.takenB && w.offB == 0;
        low.bottom = low.mine && (kDepth > 9 || 2 * j <= kSize);
        low.at[0] = at8(w);
#pragma unroll
        for (int L = 9; L <= kEnd; ++L) {
            const int4 p = pair(kind(L), 2 * j, low.bottom);
            if (L == 9) {
                __builtin_amdgcn_sched_barrier(0);
                beside();
            }
            const bool right = p.z > p.x && !(kDepth == 9 && 2 * j == kSize);
            low.at[L - 8] = {right ? p.z : p.x, right ? p.w : p.y};
            j = 2 * j + right;
        }
        low.j = j;
        return low;
    }
    // The new entry rises from a long list's leaf.  Below the registers every
    // entry of the path is written back, moved or not, which needs no branch
    // (in device memory: only where it moves); most entries stay there, and the
    // registers are left alone.
    __device__ __forceinline__ void rise(const Path &w, const Low &low, int k, int v, int lane) {
        if (kOneLast) {
            Cell last = J;
            const Cell &up = low.at[kEnd - 8];
            take(last, up, k, up.k > k ? up.v : v);
            J = pick(low.mine && 2 * low.j == kSize, last, J);
        }
#pragma unroll
        for (int L = kEnd; L >= 9; --L) {
            const Cell &own = low.at[L - 8], &up = low.at[L - 9];
            const bool moves = own.k > k, down = up.k > k;
            put(kind(L), low.j >> (kEnd - L), min(own.k, max(up.k, k)),
                moves ? down ? up.v : v : own.v, low.bottom && (kind(L) == 3 || moves));
        }
        if (__ballot(low.mine && low.at[0].k > k)) shift(w, parents(lane), k, v, lane);
    }
    // The key of the leaf, for push_entries().
    __device__ __forceinline__ int leaf_key(const Path &w, const Low &low, int lane) const {
        int x = kBelowAll;
        if (kLong) {
            x = low.bottom ? low.at[kEnd - 8].k : low.at[0].k;
            if (kOneLast) x = 2 * low.j == kSize ? J.k : x;
            x = low.mine ? x : kBelowAll;
        } else {
            // the largest key of the path
            const Spread t = on<true>(w, kAboveAll, kBelowAll, lane);
            x = min(A.k, t.A);
            if (kDepth >= 6) x = max(x, min(B.k, t.B));
            if (kDepth >= 7) x = max(x, max(min(C.k, t.C), min(D.k, t.D)));
            if (kDepth >= 8) x = max(x, min(E.k, t.E));
            if (kDepth >= 8 && kLast > 0)
                x = max(max(x, min(F.k, t.F)), max(min(G.k, t.G), min(I.k, t.I)));
            if (kSize == 512) x = max(x, min(J.k, t.J));
        }
        return wave_max_key(x);
    }
    template <class WORK>
    __device__ __forceinline__ void insert(int k, int v, int lane, const WORK &beside) {
        if constexpr (kLong) {
            const Path w = path<true>();
            rise(w, walk(w, lane, beside), k, v, lane);
        } else {
            const Parents up = parents(lane);
            __builtin_amdgcn_sched_barrier(0);
            const Path w = path<true>();
            beside();
            shift(w, up, k, v, lane);
        }
    }
    // The same; returns whether the entry got in.
    __device__ __forceinline__ bool push(int k, int v, int lane) {
        if constexpr (kLong) {
            const Path w = path<true>();
            const Low low = walk(w, lane, [] {});
            int leaf = low.bottom ? low.at[kEnd - 8].k : low.at[0].k;
            if (kOneLast) leaf = 2 * low.j == kSize ? J.k : leaf;
            if (!__ballot(low.mine && leaf > k)) return false;
            rise(w, low, k, v, lane);
            return true;
        } else {
            const Parents up = parents(lane);
            __builtin_amdgcn_sched_barrier(0);
            return __ballot(shift(path<true>(), up, k, v, lane)) != 0;
        }
    }
    // Pushes, in lane order, the entries (k, v) of the lanes in `who`, as one
    // insert after the other would.  An entry not below the leaf's key changes
    // nothing: after one that stayed out the leaf's key is looked for, and all that
    // are not below it are passed over by one comparison of all lanes.  (In
    // ascending order most stay out: the path follows the larger child, not the
    // free cells.)
    __device__ __forceinline__ void push_entries(unsigned long long who, int k, int v, int lane) {
        while (who) {
            const int j = __builtin_ctzll(who);
            who &= who - 1;
            if (push(rl(k, j), rl(v, j), lane)) continue;
            const Path w = path<true>();
            Low low = {};
            if constexpr (kLong) low = walk(w, lane, [] {});
            const unsigned long long in = who & __ballot(k < leaf_key(w, low, lane));
            if (!in) return;
            who &= ~0ull << __builtin_ctzll(in);   // (those behind it meet another leaf)
        }
    }
};

// ---- result list: the H smallest distances, sorted keys per lane, entries in a log --
//
// The reference keeps them in a heap of negated keys whose root is the worst
// kept (traverse_cpu.cpp:21-39): a candidate enters iff its distance is
// strictly below that root, and replaces it.  Which array cell holds what has
// no effect on the search; only the set and its maximum do.  Here lane l owns
// S keys, largest first; the set's maximum is the
// largest first key, `holder` a lane that has it.  A candidate below the
// maximum replaces it: in the holder lane the first key leaves and the new
// key is sorted in, one v_med3_i32 per key (new[s] = the new key clamped
// between old[s + 1] and old[s]); every other lane runs the same
// instructions with the largest integer for a key, which changes nothing.
// Then a wavefront maximum over the first keys.  No key is ever looked up by
// cell, so nothing depends on S but the S clamps: 22 instructions at S = 2,
// 28 at S = 8 (cells looked up by position: 33 and 71).  Measured in the
// refine, with the entries pushed by push_entries and the next row requested
// early: 10 000 queries over 1M x 96 at H = 96 2.48 -> 2.10 ms, one query 512
// -> 451 us; 1M x 768 at H = 256, 37 queries 1.37 -> 1.14 ms.
// Which node a key belongs to is not kept here: every admitted candidate is
// also appended to a log in the wavefront's device memory (ResultLog), and
// the final set is read back from the log by its keys.
template <int S>
struct ResultKeys {
    static constexpr int kInf = 0x7f800000;          // float_to_key(+inf)
    static constexpr int kNegInf = (int)0x807fffff;  // float_to_key(-inf)
    int key[S];   // this lane's keys, key[0] >= key[1] >= ...
    int worst;    // uniform: the largest key of the set
    int holder;   // uniform: a lane whose key[0] is `worst`

    // Empty cells hold +inf (the maximum is +inf until H candidates came),
    // cells beyond H hold -inf and never win.
    __device__ __forceinline__ void init(int H, int lane) {
#pragma unroll
        for (int s = 0; s < S; ++s) key[s] = lane * S + s < H ? kInf : kNegInf;
        worst = kInf;
        holder = 0;
    }
    // Caller has checked k < worst.  In two parts for a caller that computes
    // the wavefront maximum of the first keys itself (`reduced`: any register
    // whose lane 63 holds it).
    __device__ __forceinline__ int replace_worst(int k, int lane) {
        const int kk = lane == holder ? k : 0x7fffffff;
#pragma unroll
        for (int s = 0; s + 1 < S; ++s) key[s] = med3(key[s + 1], key[s], kk);
        key[S - 1] = min(key[S - 1], kk);
        return key[0];
    }
    __device__ __forceinline__ void set_worst(int reduced) {
        worst = __builtin_amdgcn_readlane(reduced, kWave - 1);
        holder = __builtin_ctzll(__ballot(key[0] == worst));
    }
    __device__ __forceinline__ void insert(int k, int lane) {
        replace_worst(k, lane);
        worst = wave_max_key(key[0]);
        holder = __builtin_ctzll(__ballot(key[0] == worst));
    }
};

// The log behind ResultKeys: (key, value) of every admitted candidate, in the
// wavefront's device memory.  An entry whose key is below the set's maximum
// is in the set (an entry leaves the set as its maximum, and the maximum only
// falls); entries at the maximum are in it or tie with one that is, at most H
// of them at any time.  So cutting the log down to the entries at or below
// the maximum leaves fewer than 2H, and a log of 2H + 128 entries always has
// room for the 64 candidates of a step after a cut.
struct ResultLog {
    int2 *entry;   // device memory, capacity entries, 8-byte aligned
    int n;         // uniform: entries in use
    int capacity;  // uniform

    __host__ __device__ static constexpr int capacity_for(int H) { return 2 * H + 128; }

    // Lanes whose bit is set in `who` append (k, v), in lane order.
    __device__ __forceinline__ void append(unsigned long long who, int k, int v,
                                           int lane) {
        if ((who >> lane) & 1) entry[n + lane_rank(who)] = make_int2(k, v);
        n += __popcll(who);
    }
    // The wavefront's own stores must be visible to the loads of its other
    // lanes: both go through the compute unit's cache, program order and a
    // wait for the stores are enough.
    __device__ __forceinline__ static void settle() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    }
    // Drops the entries above `worst`, in place, order kept.
    __device__ __forceinline__ void cut(int worst, int lane) {
        settle();
        int m = 0;
        for (int base = 0; base < n; base += kWave) {
            const int i = base + lane;
            int2 e = make_int2(0x7fffffff, -1);
            if (i < n) e = entry[i];
            const bool keep = i < n && e.x <= worst;
            const unsigned long long mask = __ballot(keep);
            // m + rank <= i: the write lands on an entry already read
            if (keep) entry[m + lane_rank(mask)] = e;
            m += __popcll(mask);
        }
        n = m;
        settle();
    }
    __device__ __forceinline__ bool nearly_full() const { return n > capacity - kWave; }
};

// ---- visited set ----------------------------------------------------------------
//
// Exact, like the reference's per-query marks (extension/inc/bitmask.hpp).  An
// LDS table of 2^LOG2 buckets of WAYS 16-bit tags remembers the nodes marked:
// node v lives in bucket v mod 2^LOG2 under the tag v / 2^LOG2 (bucket and tag
// give v back), and nothing is ever evicted.  While a bucket has a free slot,
// every node ever marked for it is in it: a miss means "never marked" and the
// node is added — no memory traffic at all.  A node that finds its bucket full
// is marked in the wavefront's slice of a pooled bitmask in device memory
// instead (atomic OR), which is exact as well; so is every node when the tags
// would not fit 16 bits.  Scattered atomics on a bitmask that does not stay
// in cache cost a random memory access each way and take bandwidth from the
// row reads; with the table they are the exception.  (The subgraph traversal
// keeps its smaller two-way table of recently marked rows in front of the
// bitmask: its bitmask slices are a quarter of the size and stay in cache,
// and the swap loop costs that kernel more than the atomics it saves —
// measured 3.6 against 3.3 ms.)
// The lanes of a wavefront mark their nodes at once: a slot is claimed with
// an LDS compare-and-swap, a lane whose swap fails looks again.
template <int LOG2, int WAYS = 4>
struct Visited {
    static_assert(WAYS % 2 == 0, "two tags per word");
    static constexpr int kBuckets = 1 << LOG2;
    static constexpr int kBucketWords = WAYS / 2;
    static constexpr int kWords = kBucketWords * kBuckets;
    uint32_t *table;  // LDS, kWords
    uint32_t *bits;   // device memory: one bit per node, zero between queries
    bool small;       // tags fit 16 bits (0xffff marks a free slot)
    bool dirty;       // this lane has set a bit in `bits`
    bool zeroed;      // uniform: `bits` has been cleared

    __device__ __forceinline__ void init(uint32_t *lds_words, uint32_t *slice,
                                         int n_nodes) {
        table = lds_words, bits = slice;
        small = n_nodes <= (0xffff << LOG2);
        dirty = zeroed = false;
    }
    __device__ __forceinline__ void reset(int lane) {
        for (int i = lane; i < kWords; i += kWave) table[i] = 0xffffffffu;
    }
    // Marks node v (>= 0) in the table.  Returns 0: it was marked before; 1: it
    // was not; 2: the bitmask has to be asked.
    __device__ __forceinline__ int probe(int v) {
        if (small) {
            const uint32_t tag = (uint32_t)v >> LOG2;
            uint32_t *w = table + kBucketWords * (v & (kBuckets - 1));
            for (;;) {
                uint32_t word[kBucketWords];
#pragma unroll
                for (int i = 0; i < kBucketWords; ++i)
                    word[i] = __hip_atomic_load(w + i, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_WAVEFRONT);
                bool found = false;
                int at = -1;  // first free slot: word at / 2, half at % 2
#pragma unroll
                for (int i = kBucketWords - 1; i >= 0; --i) {
                    found |= (word[i] & 0xffffu) == tag || (word[i] >> 16) == tag;
                    at = (word[i] >> 16) == 0xffffu ? 2 * i + 1 : at;
                    at = (word[i] & 0xffffu) == 0xffffu ? 2 * i : at;
                }
                if (found) return 0;
                if (at < 0) break;  // bucket full
                uint32_t old = word[0];
#pragma unroll
                for (int i = 1; i < kBucketWords; ++i) old = (at >> 1) == i ? word[i] : old;
                const uint32_t neu = (at & 1) ? (old & 0xffffu) | (tag << 16)
                                              : (old & 0xffff0000u) | tag;
                if (atomicCAS(w + (at >> 1), old, neu) == old) return 1;
            }
        }
        return 2;
    }
    // Whether the table alone shows that node v (>= 0) is marked (looked up
    // beside the marking: a mark may be missed, none is seen that is not there).
    __device__ __forceinline__ bool known(int v) const {
        if (!small) return false;
        const uint32_t tag = (uint32_t)v >> LOG2;
        const uint32_t *w = table + kBucketWords * (v & (kBuckets - 1));
        bool found = false;
#pragma unroll
        for (int i = 0; i < kBucketWords; ++i) {
            const uint32_t word =
                __hip_atomic_load(w + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            found |= (word & 0xffffu) == tag || (word >> 16) == tag;
        }
        return found;
    }
    // Marks the lanes' nodes v (negative: none), all lanes together; true in a
    // lane whose node was not marked before.  The slice of `words` is cleared when
    // it is asked for the first time.
    __device__ __forceinline__ bool mark(int v, int words, int lane) {
        const int state = v >= 0 ? probe(v) : 0;
        bool is_new = state == 1;
        if (__ballot(state == 2)) {
            if (!zeroed) clear(words, lane);
            zeroed = true;
            if (state == 2) {
                dirty = true;
                is_new = !((atomicOr(&bits[v >> 5], 1u << (v & 31)) >> (v & 31)) & 1u);
            }
        }
        return is_new;
    }
    __device__ __forceinline__ void clear(int words, int lane) {
        for (int w = lane * 4; w < words; w += kWave * 4)
            *reinterpret_cast<uint4 *>(bits + w) = make_uint4(0, 0, 0, 0);
        // (only this wavefront touches the slice)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    // after a query: the slice back to zero if any lane touched it
    __device__ __forceinline__ void clean(int words, int lane) {
        if (__ballot(dirty)) clear(words, lane);
        dirty = false;
    }
};

// ---- distances ---------------------------------------------------------------

// Squared L2 from the query (LDS) to the storage rows listed in cand_id[0..n),
// written to cand_key: four lanes per row, 16 rows per pass, two passes' loads
// in flight together where TWO says so (and the row length is known).  The
// second set of rows costs 4 DP8 / 2 registers: measured per 10 000 queries
// over a million rows, lists of 128 cells, 128-float rows 2.78 -> 2.73 ms
// (1024 queries 0.80 -> 0.745, one query 542 -> 526 us), 64-float rows 1.67 ->
// 1.74 ms in the traversal, whose fifth wavefront per SIMD it takes, but 0.84
// -> 0.80 ms per 3001 queries in the wide kernel, which reads more rows a step;
// there 128-float rows gain too, although three wavefronts per SIMD are left of
// five and six: pools of 32 to 512, one query 116 -> 100, 208 -> 182, 562 -> 481,
// 1468 -> 1287 us, 10 000 1.58 -> 1.52, 2.78 -> 2.69, 4.97 -> 4.81, 10.9 -> 10.6
// ms, 2048 10 000 30.5 -> 29.2 ms.  Where not: make_plan and pick_wide_dp.
template <int DP8, bool TWO>
__device__ __forceinline__ void eval_rows(const float *__restrict__ storage,
                                          const float *qv, const int *cand_id,
                                          float *cand_key, int n, int dp,
                                          int lane) {
    const int quad = lane >> 2, part = lane & 3;
    const float2 *qq = reinterpret_cast<const float2 *>(qv) + part * query_run(dp >> 3);
    int base = 0;
    if constexpr (TWO && DP8 > 0 && DP8 % 2 == 0) {
        for (; base + kRowsPerPass < n; base += 2 * kRowsPerPass) {
            const int c = base + quad, c2 = c + kRowsPerPass;
            const bool two = c2 < n;
            const float *row = storage + (size_t)cand_id[c] * (size_t)dp;
            const float *row2 = row;
            if (two) row2 = storage + (size_t)cand_id[c2] * (size_t)dp;
            float s, s2;
            quad_square_dist_two_rows<DP8>(row, row2, qq, part, two, s, s2);
            if (part == 0) {
                cand_key[c] = s;
                if (two) cand_key[c2] = s2;
            }
        }
    }
    for (; base < n; base += kRowsPerPass) {
        const int c = base + quad;
        const bool active = c < n;
        const float *row = storage;
        if (active) row = storage + (size_t)cand_id[c] * (size_t)dp;
        const float s = quad_square_dist_rows<DP8>(row, qq, dp >> 3, part, active);
        if (active && part == 0) cand_key[c] = s;
    }
}

// The lanes that `wanted` names first, in order, then the others.
struct LaneRows {
    int n;     // wanted
    int id;    // lane c: the id of the c-th
    int from;  // and its lane
    __device__ __forceinline__ LaneRows(bool wanted, int x, int lane) {
        const unsigned long long mask = __ballot(wanted);
        n = __popcll(mask);
        const int to4 = (wanted ? lane_rank(mask) : n + lane_rank(~mask)) << 2;
        id = __builtin_amdgcn_ds_permute(to4, x);
        from = __builtin_amdgcn_ds_permute(to4, lane);
    }
    __device__ __forceinline__ static int of(int x, int c) {
        return __builtin_amdgcn_ds_bpermute(c << 2, x);
    }
};

// The same for the rows of lanes that `wanted` names, the distance of lane l's row
// to dist[l] (LDS).
template <int DP8, bool TWO>
__device__ __forceinline__ void eval_lanes(const float *__restrict__ storage, const float *qv,
                                           bool wanted, int id, float *dist, int dp, int lane) {
    const LaneRows rows(wanted, id, lane);
    const int n = rows.n, row_id = rows.id, from = rows.from;
    const int quad = lane >> 2, part = lane & 3;
    const float2 *qq = reinterpret_cast<const float2 *>(qv) + part * query_run(dp >> 3);
    auto of = [](int x, int c) { return LaneRows::of(x, c); };
    int base = 0;
    if constexpr (TWO && DP8 > 0 && DP8 % 2 == 0) {
        for (; base + kRowsPerPass < n; base += 2 * kRowsPerPass) {
            const int c = base + quad, c2 = c + kRowsPerPass;
            const bool two = c2 < n;
            const int id1 = of(row_id, c), id2 = of(row_id, c2);
            const int at1 = of(from, c), at2 = of(from, c2);
            const float *row = storage + (size_t)id1 * (size_t)dp;
            const float *row2 = two ? storage + (size_t)id2 * (size_t)dp : row;
            float s, s2;
            quad_square_dist_two_rows<DP8>(row, row2, qq, part, two, s, s2);
            if (part == 0) {
                dist[at1] = s;
                if (two) dist[at2] = s2;
            }
        }
    }
    for (; base < n; base += kRowsPerPass) {
        const int c = base + quad;
        const bool active = c < n;
        const int id1 = of(row_id, c), at1 = of(from, c);
        const float *row = active ? storage + (size_t)id1 * (size_t)dp : storage;
        const float s = quad_square_dist_rows<DP8>(row, qq, dp >> 3, part, active);
        if (active && part == 0) dist[at1] = s;
    }
}

// ---- helpers ------------------------------------------------------------------
//
// A search with the device to itself waits for memory two thirds of its time: a
// node's neighbour ids, then their rows.  More wavefronts of its workgroup do that
// for nodes it is about to expand (the top of the open list: 92 % of the popped
// nodes are its root after the pop before, 88 % were among its first seven three
// steps before).  The search puts a node into a slot in LDS, a helper that is free
// takes it from there and leaves the node's neighbours and their distances in the
// slot.  A distance depends on the row and the query alone, so work for a node
// that is not popped soon, or ever, costs time and nothing else.
//
// A slot has one writer at a time: the search while it is idle, else the helper
// that claimed it.  LDS operations of a wavefront take effect in order.  A slot
// that holds a node is always taken and finished, so every wait of the search
// ends; a helper returns at kExit, which the search gives when all are idle.
//
// With PARTS = 2 a slot is two jobs, for two helpers: the even lanes' neighbours and
// the odd lanes'.
template <int HELPERS, int PARTS = 1>
struct LookAhead {
    static constexpr int kIdle = -1, kTaken = -2, kExit = -3;   // else: the node to do
    static constexpr bool kEarlyIds = PARTS == 2;    // ids() is called before take()
    static constexpr int kUnset = (int)0x80000000;   // a neighbour not there yet
    static constexpr int kSlots = HELPERS > 0 ? 8 : 1;
    static constexpr int kJobs = kSlots * PARTS;   // of slot s: s, s + kSlots
    static_assert(PARTS == 1 || PARTS == 2, "see slots_idle()");
    // Set in the open list's value of a node that has been put into a slot.
    static constexpr int kAsked = 1 << 30;
    static constexpr unsigned long long kTop = 0xfe;   // its first seven cells
    struct Slots {
        int job[kJobs];
        int ids[kSlots][HELPERS > 0 ? kWave : 4];
        float dist[kSlots][HELPERS > 0 ? kWave : 4];
    };
    Slots &slots;
    int node;    // lane s: what slot s holds or will hold, until it is taken; -1
    int ring;    // the slot used next (the one used longest ago)
    unsigned long long idle;   // slots seen idle since they were last used

    template <class T>
    __device__ __forceinline__ static T get(const T &x) {
        return __hip_atomic_load(&x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ static void put(int &x, int value) {
        __hip_atomic_store(&x, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    // LDS operations before this come before those after it.
    __device__ __forceinline__ static void in_order() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }

    template <class WORK>
    __device__ __forceinline__ static void help(Slots &slots, int lane, WORK &&work) {
        for (;;) {
            const int job = get(slots.job[lane & (kJobs - 1)]);
            if (__ballot(job == kExit)) return;
            const unsigned long long todo = __ballot(job >= 0);
            if (!todo) {
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            const int mine = __builtin_ctzll(todo) & (kJobs - 1);
            const int node = __builtin_amdgcn_readlane(job, mine);
            int was = node;
            if (lane == 0) was = atomicCAS(&slots.job[mine], node, kTaken);
            if (uni(was) != node) continue;   // another helper was first
            in_order();
            const int slot = mine & (kSlots - 1);
            work(node, mine, slots.ids[slot], slots.dist[slot]);
            in_order();
            if (lane == 0) put(slots.job[mine], kIdle);
        }
    }

    // What a helper does before it reads rows, in this order: look which neighbours
    // are marked, have the answers, and only then show the search their numbers.
    // The search marks what ids() gives it at once, before it takes the distances: a
    // helper that looked after that would take the node's own marks for older ones
    // and leave distances out that the search is about to use.  `v`: the lane's
    // neighbour, -1 for none; `mine`: it is of this helper's part.  Returns whether the
    // lane's row is to be read.  (Of functions, so that a test can stand between them.)
    template <class MARKED, class ANSWERED, class SHOW>
    __host__ __device__ __forceinline__ static bool look_then_show(int v, bool mine,
                                                                   const MARKED &marked,
                                                                   const ANSWERED &answered,
                                                                   const SHOW &show) {
        const bool wanted = mine && v >= 0 && !marked(v);
        answered();
        if (mine) show(v);
        return wanted;
    }

    // (bits 0 .. kSlots - 1 count)
    __device__ __forceinline__ static unsigned long long slots_idle(int job) {
        const unsigned long long jobs = __ballot(job == kIdle);
        return PARTS == 2 ? jobs & jobs >> kSlots : jobs;
    }
    __device__ __forceinline__ void look(int lane) {
        idle = slots_idle(get(slots.job[lane & (kJobs - 1)]));
    }
    // Nothing is asked for; all slots are idle.
    __device__ __forceinline__ void begin(int lane) {
        in_order();   // what the helpers are to read is in LDS
        node = -1, ring = 0;
        look(lane);
    }
    // The next slot is idle.
    __device__ __forceinline__ bool room() const { return (idle >> ring) & 1; }
    // Puts `what` into it; returns the node it held that was not taken, or -1.
    __device__ __forceinline__ int give(int what, int lane) {
        const int old = __builtin_amdgcn_readlane(node, ring);
        node = lane == ring ? what : node;
        if (kEarlyIds) put(slots.ids[ring][lane], kUnset);
        // (not the other way round, also not by the compiler: a helper's neighbours would
        // be unset again, and ids() would wait for them for ever)
        asm volatile("" ::: "memory");
        if (PARTS == 1 ? lane == ring : lane < kJobs && (lane & (kSlots - 1)) == ring)
            put(slots.job[lane], what);
        idle &= ~(1ull << ring);
        ring = (ring + 1) & (kSlots - 1);
        return old;
    }
    // Puts the first node at the top of the open list (its bank A) that is in no
    // slot into one.  One whose slot that was may be put into one again.
    __device__ __forceinline__ void ask(int &top, int lane) {
        const unsigned long long open =
            __ballot((unsigned)top < (unsigned)kAsked) & kTop;
        if (!open || !room()) return;
        const int at = __builtin_ctzll(open);
        const int old = give(__builtin_amdgcn_readlane(top, at), lane);
        top = lane == at ? top | kAsked : top;
        top = top == (old | kAsked) && old >= 0 ? old : top;
    }
    // Puts the node whose key is the lowest into a slot, if there is room: the
    // entries' best are known before the list is made of them.  `value`: by lane, the
    // node or what is below 0; the one put is flagged in it.
    __device__ __forceinline__ void ask_lowest(int key, int &value, int lane) {
        const int best = ~wave_max_key(~((unsigned)value < (unsigned)kAsked ? key : 0x7fffffff));
        const unsigned long long at = __ballot((unsigned)value < (unsigned)kAsked && key == best);
        if (!at || !room()) return;
        const int l = __builtin_ctzll(at);
        give(__builtin_amdgcn_readlane(value, l), lane);
        value = lane == l ? value | kAsked : value;
    }
    // What the slot of the node popped holds: its neighbours (by lane, -1: none)
    // and the distances of those that were not marked yet when it was asked for.
    // All of it is read at once when the node is known, in the hope that the helper
    // is done (`job`, read before the rest), so that it travels beside the pop.
    // Then take() waits for all of it, or, where rows are long and marking takes
    // time, ids() for the neighbours alone, which are there before their rows are
    // read, and take() later (short rows: 128 queries, 32 floats, 372 us without ids(),
    // 401 with it).
    struct Found {
        int slot, job, id;
        float dist;
    };
    __device__ __forceinline__ void read(Found &f, int lane) const {
        f.job = get(slots.job[lane & (kJobs - 1)]);
        asm volatile("" ::: "memory");
        f.id = get(slots.ids[f.slot][lane]);
        f.dist = get(slots.dist[f.slot][lane]);
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ Found find(int what, int lane) {
        Found f;
        unsigned long long has = __ballot(node == what);
        if (!has) {
            while (!room()) look(lane);
            has = 1ull << ring;
            give(what, lane);
        }
        f.slot = __builtin_ctzll(has) & (kSlots - 1);
        node = node == what ? -1 : node;
        read(f, lane);
        __builtin_amdgcn_sched_barrier(0);
        return f;
    }
    // Come after find() and, the first that is called, before the next give().
    __device__ __forceinline__ void ids(Found &f, int lane) {
        static_assert(kEarlyIds, "the slots' neighbours are unset when they are given");
        idle = slots_idle(f.job);
        while (__ballot(f.id == kUnset)) f.id = get(slots.ids[f.slot][lane]);
    }
    __device__ __forceinline__ void take(Found &f, int lane) {
        unsigned long long there = slots_idle(f.job);
        if (!kEarlyIds) idle = there;
        while (!((there >> f.slot) & 1)) {
            read(f, lane);
            idle = there = slots_idle(f.job);
        }
        in_order();   // read before the slot is used again
    }
    // All slots are idle.
    __device__ __forceinline__ void drain(int lane) {
        do look(lane);
        while (~idle & ((1ull << kSlots) - 1));
        asm volatile("" ::: "memory");   // (what helpers read is not changed before)
    }
    // A job for every helper, 0 .. HELPERS - 1 (all slots are idle), whose results
    // have a place of their own.
    __device__ __forceinline__ void give_all(int what, int lane) const {
        static_assert(HELPERS <= kJobs, "a job for every helper");
        in_order();
        if (lane < HELPERS) put(slots.job[lane], what);
    }
    __device__ __forceinline__ void end(int lane) const {
        if (lane < kJobs) put(slots.job[lane], kExit);
    }
};

}  // namespace pa

#endif
