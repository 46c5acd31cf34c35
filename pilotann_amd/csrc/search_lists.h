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

// ---- open list: heapq.cuh, top of the heap in registers ----------------------
//
// The reference's open list is an array heap of 2H cells with the sift rules
// of extension/inc/heapq.cuh:13-88.  Here node i of that array is node
// j = i + 1 (children 2j and 2j + 1), level L holds j in [2^L, 2^(L+1)).
//
// Levels 0..7 live in registers, one node per lane: bank A levels 0..5 (node j
// in lane j), bank B level 6 (lane j - 64), banks C and D the left and right
// children of level 7 (lane (j - 128) / 2), so a sibling pair is always two
// v_readlane of known registers.  Deeper nodes sit in LDS at [j - 256] as
// (key, value), a sibling pair per aligned 16 bytes; with DEEP the levels
// from DEEP on sit in device memory instead (the wavefront's own region, at
// [j - 2^DEEP], same cells): a long list then takes less LDS, more
// wavefronts fit a compute unit, and a walk pays one memory round trip per
// such level.  Keys are kept as
// order-preserving integers (float_to_key) so that every comparison of a walk
// is a scalar integer compare.  All lanes run the same, uniform, control flow; the walks
// are unrolled by level so that each level is a dozen instructions.  After
// each operation the heap is, cell for cell, the reference's.  Every lane
// stores the same values to the same LDS cells and reads the same cells, so a
// lane only ever reads back its own stores and the walks need no fences.
__device__ __forceinline__ int float_to_key(float x) {
    const int b = __float_as_int(x);
    return b ^ ((b >> 31) & 0x7fffffff);
}
__device__ __forceinline__ float key_to_float(int k) {
    return __int_as_float(k ^ ((k >> 31) & 0x7fffffff));
}

// c + (a != b) on the scalar unit (the compiler routes the boolean of a
// uniform compare through a vector register otherwise).
__device__ __forceinline__ int add_if_ne(int c, int a, int b) {
    int r;
    asm("s_cmp_lg_u32 %1, %2\n\ts_addc_u32 %0, %3, 0"
        : "=s"(r)
        : "s"(a), "s"(b), "s"(c)
        : "scc");
    return r;
}

constexpr int floor_log2(int x) { return x <= 1 ? 0 : 1 + floor_log2(x >> 1); }

// c + bit `idx` of a 64-bit lane mask, on the scalar unit.
__device__ __forceinline__ int add_if_bit(int c, unsigned long long mask, int idx) {
    int r;
    asm("s_bitcmp1_b64 %1, %2\n\ts_addc_u32 %0, %3, 0"
        : "=s"(r)
        : "s"(mask), "s"(idx), "s"(c)
        : "scc");
    return r;
}

// Cells of an open list of 2H cells that sit in device memory when the levels
// from `deep` on do (0: none do).
constexpr int open_list_deep_cells(int H, int deep) {
    return deep >= 8 && deep <= floor_log2(2 * H) ? 2 * H + 2 - (1 << deep) : 0;
}

template <int H, int DEEP = 0>
struct OpenList {
    static constexpr int kSize = 2 * H;           // cells of the reference heap
    static constexpr int kDepth = floor_log2(kSize);  // deepest level
    static constexpr int kRegNodes = 256;
    static constexpr int kDeepCells = open_list_deep_cells(H, DEEP);
    static constexpr int kDeepFrom = kDeepCells ? DEEP : kDepth + 1;
    static constexpr int kDeepBase = 1 << kDeepFrom;  // first node in device memory
    static constexpr int kLdsCells =
        kDeepCells ? kDeepBase - kRegNodes
                   : (kSize + 2 > kRegNodes ? kSize + 2 - kRegNodes : 0);
    static constexpr int kInf = 0x7f800000;       // float_to_key(+inf)
    static constexpr int kBelowAll = (int)0x80000000;
    static constexpr int kRegLevels = kDepth < 7 ? kDepth : 7;
    static constexpr int kLow = kDepth - kRegLevels;  // levels below the registers
    int Ak, Av, Bk, Bv, Ck, Cv, Dk, Dv;
    int2 *cells;  // node j in [256, kDeepBase) at [j - 256] as (key, value); 16-byte aligned
    int2 *deep;   // node j >= kDeepBase at [j - kDeepBase], device memory, 16-byte aligned
    int4 pending;   // pop(): the requested pair of level kDeepFrom, until pop_finish()
    int pending_j;  // its parent, 0 = nothing pending (uniform)

    __device__ __forceinline__ static int rl(int x, int l) {
        return __builtin_amdgcn_readlane(x, l);
    }
    // the value of another lane of a bank (taken modulo 64)
    __device__ __forceinline__ static int of_lane(int bank, int l) {
        return __builtin_amdgcn_ds_bpermute(l << 2, bank);
    }
    // A path from the root is named by its node on level 7, or by the
    // leftmost descendant there of the node it ends in: the path's node on
    // level L is at7 >> (7 - L).  For bank A: 7 - the level of the lane's node
    // (lane 0, which holds none: 1, where no path matches).
    __device__ __forceinline__ static int above7(int lane) {
        return lane ? __builtin_clz(lane) - 24 : 1;
    }
    // storage class of a level: 0 bank A, 1 bank B, 2 banks C/D, 3 LDS,
    // 4 device memory
    __device__ __forceinline__ static constexpr int kind(int level) {
        return level <= 5 ? 0 : level == 6 ? 1 : level == 7 ? 2
                                           : level < kDeepFrom ? 3 : 4;
    }

    __device__ __forceinline__ void reset(int lane) {
        Ak = lane == 0 ? kBelowAll : kInf;  // lane 0 holds no node: the root's parent
        Bk = Ck = Dk = kInf;
        Av = Bv = Cv = Dv = -1;
        for (int i = lane; i < kLdsCells; i += kWave) cells[i] = make_int2(kInf, -1);
        for (int i = lane; i < kDeepCells; i += kWave) deep[i] = make_int2(kInf, -1);
        pending_j = 0;
    }

    // keys (and values) of the sibling pair (c, c + 1), c even, of a level.
    // KIND and VALS are constants once the level loops are unrolled.
    __device__ __forceinline__ void pair(const int KIND, const bool VALS, int c,
                                         int &ka, int &kb, int &va,
                                         int &vb) const {
        if (KIND == 0) {
            ka = rl(Ak, c), kb = rl(Ak, c + 1);
            if (VALS) va = rl(Av, c), vb = rl(Av, c + 1);
        } else if (KIND == 1) {
            const int l = c - 64;
            ka = rl(Bk, l), kb = rl(Bk, l + 1);
            if (VALS) va = rl(Bv, l), vb = rl(Bv, l + 1);
        } else if (KIND == 2) {
            const int l = (c - 128) >> 1;
            ka = rl(Ck, l), kb = rl(Dk, l);
            if (VALS) va = rl(Cv, l), vb = rl(Dv, l);
        } else {
            // one 16-byte read: both children with their values
            const int4 p = KIND == 3
                ? *reinterpret_cast<const int4 *>(cells + (c - kRegNodes))
                : *reinterpret_cast<const int4 *>(deep + (c - kDeepBase));
            if (VALS) va = uni(p.y), vb = uni(p.w);
            ka = uni(p.x), kb = uni(p.z);
        }
    }
    __device__ __forceinline__ int key_of(const int KIND, int j) const {
        if (KIND == 0) return rl(Ak, j);
        if (KIND == 1) return rl(Bk, j - 64);
        if (KIND == 2) {
            // both banks are read and one result is kept: two instructions
            // more than a branch on the parity of j would need, no branch
            const int l = (j - 128) >> 1;
            const int left = rl(Ck, l), right = rl(Dk, l);
            return (j & 1) ? right : left;
        }
        return uni(KIND == 3 ? cells[j - kRegNodes].x : deep[j - kDeepBase].x);
    }
    __device__ __forceinline__ int val_of(const int KIND, int j) const {
        if (KIND == 0) return rl(Av, j);
        if (KIND == 1) return rl(Bv, j - 64);
        if (KIND == 2) {
            const int l = (j - 128) >> 1;
            const int left = rl(Cv, l), right = rl(Dv, l);
            return (j & 1) ? right : left;
        }
        return uni(KIND == 3 ? cells[j - kRegNodes].y : deep[j - kDeepBase].y);
    }
    // lane l of a key bank and of its value bank := two uniform values
    // (v_writelane takes one scalar register besides M0, which holds the lane)
    __device__ __forceinline__ static void set_lane(int &kbank, int &vbank, int k,
                                                    int v, int l) {
        asm("s_mov_b32 m0, %4\n\t"
            "s_nop 0\n\t"
            "v_writelane_b32 %0, %2, m0\n\t"
            "v_writelane_b32 %1, %3, m0"
            : "+v"(kbank), "+v"(vbank)
            : "s"(k), "s"(v), "s"(l)
            : "m0");
    }
    __device__ __forceinline__ void put(const int KIND, int j, int k, int v,
                                        int lane) {
        if (KIND == 0) {
            set_lane(Ak, Av, k, v, j);
        } else if (KIND == 1) {
            set_lane(Bk, Bv, k, v, j - 64);
        } else if (KIND == 2) {
            // lane-masked selects on both banks instead of a branch on the
            // parity of j around two v_writelane
            const int l = (j - 128) >> 1;
            const bool here = lane == l;
            const bool right = j & 1;
            Ck = (here && !right) ? k : Ck;
            Cv = (here && !right) ? v : Cv;
            Dk = (here && right) ? k : Dk;
            Dv = (here && right) ? v : Dv;
        } else if (KIND == 3) {
            // every lane stores the same pair to the same cell: one LDS
            // write, and no divergent branch around it
            cells[j - kRegNodes] = make_int2(k, v);
        } else {
            deep[j - kDeepBase] = make_int2(k, v);
        }
    }

    // Which child a walk takes, for every sibling pair of the register levels
    // at once: lane-parallel compares against the sibling (one DPP move per
    // bank), read back as lane masks, so that a level of the walk is three
    // scalar instructions and no register read.  LARGER selects the rule of
    // heap_replace (strictly larger right child), else that of the sift of a
    // pop (strictly smaller right child); left wins ties in both.  In banks A
    // and B bit i of the mask tells about the pair whose right child sits in
    // lane i; in banks C/D lane i holds both children.
    struct Choice {
        unsigned long long a, b, cd;
    };
    template <bool LARGER>
    __device__ __forceinline__ Choice choices() const {
        Choice ch;
        const int sa = __builtin_amdgcn_update_dpp(Ak, Ak, 0xB1, 0xF, 0xF, false);
        ch.a = __ballot(LARGER ? Ak > sa : Ak < sa);
        ch.b = 0, ch.cd = 0;
        if (kDepth >= 6) {
            const int sb = __builtin_amdgcn_update_dpp(Bk, Bk, 0xB1, 0xF, 0xF, false);
            ch.b = __ballot(LARGER ? Bk > sb : Bk < sb);
        }
        if (kDepth >= 7) ch.cd = __ballot(LARGER ? Dk > Ck : Dk < Ck);
        return ch;
    }
    // the child of j the walk takes on register level L (1..7), L < kDepth
    // or the pair is known to be complete: 2j + (bit of the pair in the
    // level's mask), three scalar instructions.  s_bitcmp1_b64 looks at the
    // low six bits of its index only, so node numbers serve as lane numbers
    // (bank B holds node j in lane j - 64, banks C/D the children of node j
    // in lane j - 64).
    __device__ __forceinline__ int step_down(const int L, int j,
                                             const Choice &ch) const {
        int r;
        if (kind(L) <= 1) {
            // t = 2j + 1, the right child, whose lane holds the pair's bit
            asm("s_lshl1_add_u32 %0, %1, 1\n\t"
                "s_bitcmp1_b64 %2, %0\n\t"
                "s_addc_u32 %0, %0, -1"
                : "=&s"(r)
                : "s"(j), "s"(kind(L) == 0 ? ch.a : ch.b)
                : "scc");
        } else {
            asm("s_lshl_b32 %0, %1, 1\n\t"
                "s_bitcmp1_b64 %2, %1\n\t"
                "s_addc_u32 %0, %0, 0"
                : "=&s"(r)
                : "s"(j), "s"(ch.cd)
                : "scc");
        }
        return r;
    }

    // heapq.cuh:37-45 with the sift of :13-29: the root leaves, (inf, -1)
    // sinks along the smaller child (left on ties).  The reference stops when
    // that child is (inf, -1) too; going on to the bottom instead only copies
    // (inf, -1) over (inf, -1) — every infinite cell carries -1 — so the
    // final state is the same and the walk is straight-line code.  Levels
    // 1..kDepth-1 are complete; on level kDepth only nodes up to kSize exist
    // and node kSize has no sibling (its absent sibling's cell holds +inf and
    // is never the smaller one).
    __device__ __forceinline__ void pop(int lane, int &out_k, int &out_v) {
        out_k = rl(Ak, 1);
        out_v = rl(Av, 1);
        const Choice ch = choices<false>();
        // The path through the register levels first (masks only); then every
        // lane on it takes the entry of its child on the path, all levels at
        // once: a lane gather from bank A (levels 0..4) and one from bank B
        // (level 5), and bank B's children are in banks C/D of the same lane.
        int j = 1;
        bool cut = false;  // level kDepth has no node below j
#pragma unroll
        for (int L = 1; L <= kRegLevels; ++L) {
            if (L == kDepth && 2 * j > kSize) cut = true;
            else j = step_down(L, j, ch);
        }
        {
            const int level = cut ? kRegLevels - 1 : kRegLevels;  // of j
            const int at7 = j << (7 - level);
            const int sh = above7(lane);
            const int child = at7 >> (sh - 1);
            bool here = (at7 >> sh) == lane;
            if (kDepth <= 6) here = here && lane < (1 << level);
            int ck = of_lane(Ak, child), cv = of_lane(Av, child);
            if (kDepth >= 6) {
                const int bk = of_lane(Bk, child), bv = of_lane(Bv, child);
                ck = lane >= 32 ? bk : ck;
                cv = lane >= 32 ? bv : cv;
            }
            if (kDepth >= 7) {
                bool hereB = lane == (at7 >> 1) - 64;
                if (kDepth == 7) hereB = hereB && !cut;
                const bool right = Dk < Ck;
                Bk = hereB ? (right ? Dk : Ck) : Bk;
                Bv = hereB ? (right ? Dv : Cv) : Bv;
            }
            Ak = here ? ck : Ak;
            Av = here ? cv : Av;
        }
        if (cut) {
            put(kind(kRegLevels - 1), j, kInf, -1, lane);
            return;
        }
        pending_j = 0;
#pragma unroll
        for (int L = kRegLevels + 1; L <= kDepth; ++L) {
            if (L == kDepth && 2 * j > kSize) {
                put(kind(L - 1), j, kInf, -1, lane);
                return;
            }
            if (kDeepCells && L == kDeepFrom) {
                // the pair is requested; pop_finish() goes on from here
                pending = *reinterpret_cast<const int4 *>(deep + (2 * j - kDeepBase));
                pending_j = j;
                return;
            }
            int ka, kb, va, vb;
            pair(kind(L), true, 2 * j, ka, kb, va, vb);
            if (L == kDepth) kb = 2 * j == kSize ? ka : kb;
            const int k = min(ka, kb);
            const int v = k != ka ? vb : va;
            const int c = add_if_ne(2 * j, k, ka);
            put(kind(L - 1), j, k, v, lane);
            j = c;
        }
        put(kind(kDepth), j, kInf, -1, lane);
    }
    // The levels of a pop that sit in device memory.  pop() only requests the
    // first pair it needs from there; the caller puts the work that does not
    // touch the list (the root is in registers) between the two, and calls
    // this before the next walk or pop.  Nothing to do without such levels.
    __device__ __forceinline__ void pop_finish(int lane) {
        if (!kDeepCells) return;
        int j = pending_j;
        if (j == 0) return;
        pending_j = 0;
#pragma unroll
        for (int L = kDeepFrom; L <= kDepth; ++L) {
            if (L == kDepth && 2 * j > kSize) {
                put(kind(L - 1), j, kInf, -1, lane);
                return;
            }
            int ka, kb, va, vb;
            if (L == kDeepFrom) {
                ka = uni(pending.x), va = uni(pending.y);
                kb = uni(pending.z), vb = uni(pending.w);
            } else {
                pair(kind(L), true, 2 * j, ka, kb, va, vb);
            }
            if (L == kDepth) kb = 2 * j == kSize ? ka : kb;
            const int k = min(ka, kb);
            const int v = k != ka ? vb : va;
            const int c = add_if_ne(2 * j, k, ka);
            put(kind(L - 1), j, k, v, lane);
            j = c;
        }
        put(kind(kDepth), j, kInf, -1, lane);
    }

    // heapq.cuh:47-77: walk to a leaf through the larger child (left on
    // ties), overwrite it when the new key is strictly smaller, let the new
    // entry rise.  In two parts so that the caller can put independent work
    // between them: the walk is straight-line code, the rise branches.
    struct Leaf {
        int j;       // the leaf
        int key;     // its key
        bool bottom; // it is on level kDepth
        // the entries of the path on levels 8 and down, as the walk read them
        int low_key[kLow ? kLow : 1], low_val[kLow ? kLow : 1];
    };
    __device__ __forceinline__ Leaf walk_to_large_leaf() const {
        return walk_below(choices<true>(), 0, 1);
    }
    // The walk from node j on level DONE down to a leaf (the levels above
    // were taken elsewhere).
    __device__ __forceinline__ Leaf walk_below(const Choice &ch, const int DONE,
                                               int j) const {
        Leaf leaf;
        bool bottom = true;  // the walk reached level kDepth
        int walked_key = 0;  // key of node j when its level is an LDS level
#pragma unroll
        for (int L = DONE + 1; L <= kDepth; ++L) {
            if (L == kDepth && 2 * j > kSize) {
                bottom = false;
                break;
            }
            if (kind(L) <= 2) {
                // node kSize has no sibling: the left child it is
                j = (L == kDepth && 2 * j == kSize) ? 2 * j : step_down(L, j, ch);
            } else {
                int ka, kb, va, vb;
                pair(kind(L), true, 2 * j, ka, kb, va, vb);
                if (L == kDepth) kb = 2 * j == kSize ? ka : kb;
                walked_key = max(ka, kb);
                leaf.low_key[L - 8] = walked_key;
                leaf.low_val[L - 8] = walked_key != ka ? vb : va;
                j = add_if_ne(2 * j, walked_key, ka);
            }
        }
        // the leaf's key: the walk has it already when the leaf is in LDS
        leaf.j = j, leaf.bottom = bottom;
        if (bottom)
            leaf.key = kind(kDepth) >= 3 ? walked_key : key_of(kind(kDepth), j);
        else
            leaf.key = kind(kDepth - 1) >= 3 ? walked_key : key_of(kind(kDepth - 1), j);
        return leaf;
    }
    // The seven register levels of that walk (lists of 256 cells and more,
    // where they are complete) together with a wavefront maximum of `x`,
    // which comes back in lane 63: the six v_max_i32_dpp of the maximum each
    // need two wait states after the one before, and the three scalar
    // instructions of a level fill them, where apart they would be s_nop.
    // Returns the node on level 7.
    static constexpr bool kFusedTop = kDepth >= 8;
    __device__ __forceinline__ static int top_levels_and_wave_max(const Choice &ch,
                                                                  int &x) {
        int j, t;
        asm("s_bitcmp1_b64 %[a], 3\n\t"
            "s_addc_u32 %[j], 2, 0\n\t"
            "v_max_i32_dpp %[x], %[x], %[x] quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
            "s_lshl1_add_u32 %[j], %[j], 1\n\t"
            "s_bitcmp1_b64 %[a], %[j]\n\t"
            "s_addc_u32 %[j], %[j], -1\n\t"
            "v_max_i32_dpp %[x], %[x], %[x] quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
            "s_lshl1_add_u32 %[j], %[j], 1\n\t"
            "s_bitcmp1_b64 %[a], %[j]\n\t"
            "s_addc_u32 %[j], %[j], -1\n\t"
            "v_max_i32_dpp %[x], %[x], %[x] row_half_mirror row_mask:0xf bank_mask:0xf\n\t"
            "s_lshl1_add_u32 %[j], %[j], 1\n\t"
            "s_bitcmp1_b64 %[a], %[j]\n\t"
            "s_addc_u32 %[j], %[j], -1\n\t"
            "v_max_i32_dpp %[x], %[x], %[x] row_mirror row_mask:0xf bank_mask:0xf\n\t"
            "s_lshl1_add_u32 %[j], %[j], 1\n\t"
            "s_bitcmp1_b64 %[a], %[j]\n\t"
            "s_addc_u32 %[j], %[j], -1\n\t"
            "v_max_i32_dpp %[x], %[x], %[x] row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
            "s_lshl1_add_u32 %[j], %[j], 1\n\t"
            "s_bitcmp1_b64 %[b], %[j]\n\t"
            "s_addc_u32 %[j], %[j], -1\n\t"
            "v_max_i32_dpp %[x], %[x], %[x] row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
            "s_lshl_b32 %[t], %[j], 1\n\t"
            "s_bitcmp1_b64 %[cd], %[j]\n\t"
            "s_addc_u32 %[j], %[t], 0"
            : [j] "=&s"(j), [x] "+v"(x), [t] "=&s"(t)
            : [a] "s"(ch.a), [b] "s"(ch.b), [cd] "s"(ch.cd)
            : "scc");
        return j;
    }
    // The new entry rises: along the path to the leaf, whose keys do not fall
    // from the root down, every entry with a larger key moves one level down
    // and the new one takes the place of the highest of them.  In one of two
    // forms, of which the second leaves the register levels alone where an
    // entry does not get that far, as most of those of long lists do not:
    //  * all levels at once: a node of the path with a key above k gets its
    //    parent's entry if that is above k too, else the new one, which all
    //    lanes decide together from the lists as they were: the parents of
    //    bank A are a lane gather away, those of bank B are in lanes 32..63 of
    //    bank A, those of banks C/D in the same lane of bank B, and the walk has
    //    read the levels below;
    //  * level by level from the leaf (kByLevel, lists of 1024 cells and more),
    //    below the registers with what the walk has read, up to the level
    //    where the entry stays.
    // Measured, first form / second, over a million rows of 128 floats and 400 000
    // of 64 floats, ms: 4096 cells 10 000 queries 42.0 / 38.4 and 28.8 / 25.5, one
    // query 6.04 / 5.38 and 4.44 / 3.98; 2048 cells 10 000 queries 24.3 / 23.6 and
    // 15.6 / 14.8; 1024 cells 10 000 queries 10.64 / 10.63 and 4.84 / 4.74, one
    // query 1.69 / 1.64 and 0.91 / 0.92; 768 cells as close; 256 cells one query
    // 0.283 / 0.292 and 512 cells 0.396 / 0.412.  (Parents read again from LDS on
    // the way up, as before the first form: 4096 cells 39.8 and 27.7.)
    static constexpr bool kByLevel = kDepth >= 10;
    __device__ __forceinline__ void replace_leaf(const Leaf &leaf, int k, int v,
                                                 int lane) {
        if (k >= leaf.key) return;
        if constexpr (kByLevel) {
            int j = leaf.j;
            // one store per level: the parent's entry while it is larger than
            // the new key, the new entry where the rise stops
            auto rise = [&](const int L) -> bool {
                const int up = j >> 1;
                const int pk = L > 8 ? leaf.low_key[L - 9] : key_of(kind(L - 1), up);
                const int pv = L > 8 ? leaf.low_val[L - 9] : val_of(kind(L - 1), up);
                const bool stop = pk <= k;
                put(kind(L), j, stop ? k : pk, stop ? v : pv, lane);
                j = up;
                return stop;
            };
            if (leaf.bottom && rise(kDepth)) return;
#pragma unroll
            for (int L = kDepth - 1; L >= 1; --L)
                if (rise(L)) return;
            put(0, 1, k, v, lane);
            return;
        }
        const int depth = leaf.bottom ? kDepth : kDepth - 1;   // of the leaf
        // the path's end in the register levels, and its level
        int j7 = leaf.j, level = depth;
        if (kLow) {
            j7 >>= depth - 7;
            level = 7;
            int pk = key_of(2, j7), pv = val_of(2, j7);
#pragma unroll
            for (int L = 8; L <= kDepth; ++L) {
                if (L == kDepth && !leaf.bottom) break;
                const int own = leaf.low_key[L - 8];
                const bool down = pk > k;
                const int node = leaf.j >> (depth - L);
                if (own > k) put(kind(L), node, down ? pk : k, down ? pv : v, lane);
                pk = own, pv = leaf.low_val[L - 8];
            }
        }
        const int at7 = j7 << (7 - level);
        const int sh = above7(lane);
        const int pAk = of_lane(Ak, lane >> 1), pAv = of_lane(Av, lane >> 1);
        if (kDepth >= 6) {
            const int pBk = of_lane(Ak, 32 + (lane >> 1)), pBv = of_lane(Av, 32 + (lane >> 1));
            const int l6 = (at7 >> 1) - 64;
            if (kDepth >= 7) {
                const bool down = Bk > k;
                const int nk = down ? Bk : k, nv = down ? Bv : v;
                bool here = lane == l6;
                if (kDepth == 7) here = here && level == 7;
                const bool hereC = here && !(at7 & 1) && Ck > k;
                const bool hereD = here && (at7 & 1) && Dk > k;
                Ck = hereC ? nk : Ck;
                Cv = hereC ? nv : Cv;
                Dk = hereD ? nk : Dk;
                Dv = hereD ? nv : Dv;
            }
            const bool down = pBk > k;
            bool here = lane == l6 && Bk > k;
            if (kDepth == 6) here = here && level == 6;
            Bk = here ? (down ? pBk : k) : Bk;
            Bv = here ? (down ? pBv : v) : Bv;
        }
        const bool down = pAk > k;
        bool here = (at7 >> sh) == lane && Ak > k;
        if (kDepth <= 5) here = here && lane < (2 << level);
        Ak = here ? (down ? pAk : k) : Ak;
        Av = here ? (down ? pAv : v) : Av;
    }
    // Pushes, in lane order, the entries (k, v) of the lanes in `who`, as one
    // replace after the other would.  `leaf` is where the walk ends in the
    // list as it stands: an entry not below its key changes nothing, so the
    // walk is taken again only after an entry that got in, and everything
    // that stays out is passed over by one comparison of all lanes.  Entries
    // mostly come in ascending order; then nearly all of them stay out (the
    // walk follows the larger child, not the free cells).
    __device__ __forceinline__ void push_entries(Leaf &leaf, unsigned long long who,
                                                 int k, int v, int lane) {
        for (;;) {
            const unsigned long long in = who & __ballot(k < leaf.key);
            if (!in) return;
            const int j = __builtin_ctzll(in);
            who &= ~1ull << j;
            replace_leaf(leaf, rl(k, j), rl(v, j), lane);
            leaf = walk_to_large_leaf();
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
    __device__ __forceinline__ static int med3(int a, int b, int c) {
        int r;
        asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
        return r;
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

    __device__ __forceinline__ void init(uint32_t *lds_words, uint32_t *slice,
                                         int n_nodes) {
        table = lds_words, bits = slice;
        small = n_nodes <= (0xffff << LOG2);
        dirty = false;
    }
    __device__ __forceinline__ void reset(int lane) {
        for (int i = lane; i < kWords; i += kWave) table[i] = 0xffffffffu;
    }
    // Marks node v (>= 0).  Returns 0: it was marked before; 1: it was not;
    // 2: the bitmask was asked, `before` will hold its word as it was (the
    // caller may look at it later, so that the atomic's round trip overlaps
    // other work): fresh() tells.
    __device__ __forceinline__ int probe(int v, uint32_t &before) {
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
        dirty = true;
        before = atomicOr(&bits[v >> 5], 1u << (v & 31));
        return 2;
    }
    __device__ __forceinline__ static bool fresh(int state, uint32_t before, int v) {
        return state == 1 || (state == 2 && !((before >> (v & 31)) & 1u));
    }
    // marks node v (>= 0); true if it was not marked before
    __device__ __forceinline__ bool mark(int v) {
        uint32_t before = 0;
        const int state = probe(v, before);
        return fresh(state, before, v);
    }
    // after a query: the slice back to zero if any lane touched it
    __device__ __forceinline__ void clean(int words, int lane) {
        if (__ballot(dirty)) {
            for (int w = lane * 4; w < words; w += kWave * 4)
                *reinterpret_cast<uint4 *>(bits + w) = make_uint4(0, 0, 0, 0);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            dirty = false;
        }
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

}  // namespace pa

#endif
