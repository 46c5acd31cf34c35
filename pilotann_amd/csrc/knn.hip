// Nearest-neighbour candidates for the graph builder, gfx950.
//
// The reference hands graph construction to a library (faiss:
// pilot_ann/utils/graphs.py:15-20,52-56); its first step everywhere is "the
// closest rows of every row".  Here that step is one kernel: half-precision
// products on the matrix cores (v_mfma_f32_32x32x16_f16, float accumulation)
// fused with the selection, so the N x N table of scores never exists in
// memory.  The caller ranks the candidates again with exact float distances.
//
// A workgroup of eight wavefronts owns 256 query rows and walks over the base
// rows 256 at a time.  Per 256 x 256 tile both operands go through LDS in
// chunks of 64 elements, loaded from memory straight into two staging
// buffers; a wavefront multiplies 128 x 64 of the tile as 4 x 2 instruction
// tiles.  score(i, j) = |x_j|^2 - 2 q_i . x_j ranks the base rows of query i
// like the squared distance does.  With tiles of this size every product
// moves 1/64 byte of operands through the memory system, and that traffic,
// not the matrix cores, sets the pace.
//
// Selection: every query row has a list of (score, id) in device memory and,
// in LDS, its length and a limit from the keep-th smallest score at the time
// the list was last cut.  A score below that bound is appended (LDS atomic
// for the position); once a list could overflow with the next tile, the
// wavefront that owns the row cuts it to its `keep` smallest (a radix
// selection over the order-preserving integer image of the scores, in
// registers) and moves the limit.  Late in the walk few scores pass.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "device_common.h"
#include "pilotann.h"

using namespace pa;

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kChunk = 64;        // contraction elements staged at a time; a
                                  // row is a whole number of chunks
// Appended entries a list may hold beyond `keep` before it must be cut.  Lists
// of 256 (a graph build's) take 384: half as many cuts as with 128, and a fifth
// more entries let in by the limit of the last one (55 000 rows against 120 000
// of 768 floats: 128 21.4, 256 15.2, 384 14.9, 512 15.4 ms).  The others, 128
// and 384: of 64 13.4 and 13.6 ms there and 19.9 and 20.8 for 100 000 rows against
// 300 000 of 96 floats, of 128 14.3 and 14.2, 22.8 and 22.5; lists of 512, 21.4 and
// 19.1, 44.1 and 37.0, keep the shorter ones for their memory (1 KB a row each).
constexpr int slack(int keep) { return keep == 256 ? 384 : 128; }
constexpr int kMaxBN = 256;       // the most base rows a tile has in any form
constexpr int kRowPad = 256;      // rows the caller's arrays are padded to

struct KnnArgs {
    const _Float16 *query, *base;
    const float *base_norm;
    float *cand_score;
    int32_t *cand_id, *cand_count;
    int64_t m, n;
    int d, n_seg;
};

__device__ __forceinline__ unsigned ordered(float x) {
    const unsigned b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float unordered(unsigned u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// The larger of two or three finite numbers (the plain instructions: fmaxf
// first rewrites every operand that could be a signalling NaN).
__device__ __forceinline__ float larger(float x, float y) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
    return r;
}
__device__ __forceinline__ float larger(float x, float y, float z) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(y), "v"(z));
    return r;
}

// Every lane's 16 bytes at `from` go to LDS, side by side from `lds_addr` (the
// same for all lanes) on.  The compiler does not know of the transfer: the
// wavefront waits with bring_wait() before a barrier makes the rows public.
__device__ __forceinline__ void bring_rows(const void *from, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off"
                 :: "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(from)
                 : "memory", "m0");
}
template <int LEFT>   // until at most LEFT of the wavefront's transfers are under way
__device__ __forceinline__ void bring_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(LEFT) : "memory");
}

// The wavefront cuts one list of `n` entries (keep < n <= keep + slack + BN)
// to its `keep` smallest, which end up in its first `keep` places, and returns
// the largest score kept.
template <int KEEP, int BN>
__device__ __forceinline__ float cut_list(float *score, int32_t *id, int n, int lane) {
    constexpr int kPerLane = (KEEP + slack(KEEP) + BN + kWave - 1) / kWave;
    unsigned u[kPerLane];
    int32_t v[kPerLane];
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
        const int e = lane + kWave * i;
        u[i] = 0x7fffffffu;   // no score: ordered() of it is the largest number
        v[i] = -1;
        if (kWave * i + kWave <= KEEP || e < n) {
            u[i] = __float_as_uint(score[e]);
            v[i] = id[e];
        }
    }
    // The KEEP-th smallest, bit by bit from the highest one in which the
    // entries differ: `bound` stays the largest value with fewer than KEEP
    // entries below it, until a value with exactly KEEP below it is met, which
    // a list of a few hundred scores has after about ten bits (of 32).
    unsigned low = 0xffffffffu, high = 0;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
        u[i] = ordered(__uint_as_float(u[i]));
        low = min(low, u[i]);
        high = u[i] != 0xffffffffu ? max(high, u[i]) : high;
    }
    low = ~((unsigned)wave_max_key((int)(~low ^ 0x80000000u)) ^ 0x80000000u);
    high = (unsigned)wave_max_key((int)(high ^ 0x80000000u)) ^ 0x80000000u;
    const int top = low == high ? -1 : 31 - __builtin_clz(low ^ high);
    unsigned bound = top < 0 ? low : low & ~((2u << top) - 1u);
    bool parted = false;   // exactly KEEP entries lie below `bound`
#pragma unroll 1
    for (int bit = top; bit >= 0 && !parted; --bit) {
        const unsigned trial = bound | (1u << bit);
        int below = 0;
#pragma unroll
        for (int i = 0; i < kPerLane; ++i) below += __popcll(__ballot(u[i] < trial));
        if (below <= KEEP) bound = trial;
        parted = below == KEEP;
    }
    int n_below = 0;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) n_below += __popcll(__ballot(u[i] < bound));
    // entries below the bound first, then entries equal to it while there is room
    int at_below = 0, at_equal = n_below;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
        const bool below = u[i] < bound;
        const bool equal = u[i] == bound;
        const unsigned long long mb = __ballot(below), me = __ballot(equal);
        const int pb = at_below + lane_rank(mb), pe = at_equal + lane_rank(me);
        if (below) {
            score[pb] = unordered(u[i]);
            id[pb] = v[i];
        } else if (equal && pe < KEEP) {
            score[pe] = unordered(u[i]);
            id[pe] = v[i];
        }
        at_below += __popcll(mb);
        at_equal += __popcll(me);
    }
    if (parted) {
        high = 0;
#pragma unroll
        for (int i = 0; i < kPerLane; ++i) high = u[i] < bound ? max(high, u[i]) : high;
        bound = (unsigned)wave_max_key((int)(high ^ 0x80000000u)) ^ 0x80000000u;
    }
    return unordered(bound);
}

// WR x WC wavefronts, each multiplying WM x WN instruction tiles of 32 x 32:
// the workgroup owns BM = 32 WR WM query rows and takes BN = 32 WC WN base
// rows per tile.
//
// The sums start at -|x_j|^2 / 2 instead of zero, so a finished sum s is
// -score / 2 and "score below the row's bound" is "s above the row's limit",
// limit = -bound / 2: one comparison per product sum, and a row's sums over
// the wavefront's columns are first reduced to their maximum.
//
// Chunks flow through a ring of staging buffers without a break between
// tiles: chunk c is multiplied out of buffer c % 2 while chunk c + 1 travels
// from memory straight into the other buffer (global_load_lds, 16 bytes a
// lane; no registers and no LDS stores in between); one barrier per chunk; the
// chunk after a tile's last is the first of the next tile.
//
// SHORT: the list starts empty and a walk of few tiles, in which most sums
// pass, is all it sees: places for a wavefront's entries are drawn row by row
// with one atomic instruction, where an atomic for every lane and sum waits for
// each result and meets others on a few words.  In a long walk few sums pass
// and that form's counting costs more than it saves.  Per launch over 768
// floats: one tile a list 90 against 52 us, 2 tiles 385 against 315, 4 tiles
// 940 against 820, 32 tiles the same, 469 tiles 14.9 against 16.6 ms.
template <int KEEP, bool SHORT, int WR, int WC, int WM, int WN>
__global__ __launch_bounds__(64 * WR * WC, (WM * WN > 8 ? 1 : 2)) void knn_kernel(KnnArgs a) {
    constexpr int kThreads = kWave * WR * WC;
    constexpr int BM = 32 * WR * WM, BN = 32 * WC * WN;
    constexpr int kStageRows = kThreads / 8;   // rows one staging step covers
    constexpr int kOwnRows = BM / (WR * WC);   // lists a wavefront looks after
    static_assert(BN <= kMaxBN && kRowPad % BM == 0 && kRowPad % BN == 0, "tile sizes");
    static_assert(kOwnRows == 32 || kOwnRows == 64, "lists per wavefront");
    static_assert(BM % kStageRows == 0 && BN % kStageRows == 0, "staging steps");
    constexpr int kCap = KEEP + slack(KEEP) + kMaxBN;  // entries a list can hold
    // a staging buffer: the chunk of the query tile, then that of the base
    // tile, rows of kRow bytes without padding.  LDS has 64 banks of four
    // bytes and serves a 16-byte read to 16 lanes at a time: 16 consecutive
    // rows are 8 pairs that share a 256-byte span, so the 16-byte piece p of
    // row r lies at place p ^ ((r / 2) % 8) of its row, and neither the loads
    // that fill the buffer nor the operand reads meet in a bank
    constexpr int kRow = kChunk * 2;
#define PA_PLACE_MIX(row_) ((unsigned)((row_) / (256 / kRow)) & (unsigned)(kPieces - 1))
    constexpr int kPieces = kRow / 16;             // 16-byte pieces of a row
    constexpr int kInstrRows = kWave / kPieces;    // rows one instruction brings
    constexpr int kStage = (BM + BN) * kRow;
    constexpr int kStages = (128 << 10) / kStage;  // buffers in the ring
    constexpr int kWaves = WR * WC;
    constexpr int kWaveRows = (BM + BN) / kWaves;  // rows a wavefront brings in per chunk
    constexpr int kInstrs = kWaveRows / kInstrRows;
    static_assert(kPieces == 8 || kPieces == 4, "chunk size");
    static_assert(kStages >= 2 && kWaveRows % kInstrRows == 0 && BM % kWaveRows == 0,
                  "rows per wavefront");
    // transfers that may still be under way when the chunk needed next must
    // be there: those of the chunks after it
    constexpr int kAhead = kInstrs * (kStages - 2);
    __shared__ __align__(1024) unsigned char stage[kStages * kStage];
    __shared__ int count[BM];
    __shared__ float limit[BM];
    const int t = threadIdx.x;
    const int lane = t & (kWave - 1), wave = t / kWave;
    const int wr = wave % WR, wc = wave / WR;
    const int col = lane & 31, half = lane >> 5;
    const int64_t q0 = (int64_t)blockIdx.x * BM;
    const int seg = blockIdx.y;
    float *my_score = a.cand_score + ((size_t)seg * a.m + q0) * kCap;
    int32_t *my_id = a.cand_id + ((size_t)seg * a.m + q0) * kCap;

    for (int r = t; r < BM; r += kThreads) {
        count[r] = 0;
        limit[r] = q0 + r < a.m ? -INFINITY : INFINITY;  // rows past the end take nothing
    }

    // staging goes from memory straight into LDS: one instruction of a
    // wavefront brings kInstrRows rows of a chunk, lane l a piece of row
    // l / kPieces, the piece that belongs at place l % kPieces, and the
    // hardware puts the lanes' 16 bytes side by side.
    // The caller's arrays are readable up to the next multiple of kRowPad
    // rows, and a row is a whole number of chunks: no clamping
    const int my_first = wave * kWaveRows;      // among the BM + BN rows of a buffer
    const bool brings_query = my_first < BM;
    const int bring_row = lane / kPieces;
    const unsigned bring_off =
        ((unsigned)((brings_query ? my_first : my_first - BM) + bring_row) * (unsigned)a.d) * 2u;
    const unsigned char *a_base =
        reinterpret_cast<const unsigned char *>(a.query) + (size_t)q0 * a.d * 2;
    const unsigned bring_to =
        (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)stage + my_first * kRow;
    // operand reads: lane l wants elements 16 s + 8 (l / 32) .. + 8 of row
    // l % 32 of an instruction tile, piece 2 s + l / 32 of that row
    const unsigned mix = PA_PLACE_MIX(col);
    const unsigned swizzle = 16u * (half ^ (mix & 1)) + 32u * (mix >> 1);
    const unsigned char *a_tile = stage + (wr * WM * 32 + col) * kRow;
    const unsigned char *b_tile = stage + (BM + wc * WN * 32 + col) * kRow;
    const int64_t n_tiles = (a.n + BN - 1) / BN;

    int64_t f_tile = seg;   // the chunk the next fetch takes: tile and element
    int f_k0 = 0;
    bool pending;           // a chunk is on its way into the other buffer
// the next chunk, if there is one, from memory into staging buffer `buf`
#define PA_FETCH_NEXT(buf)                                                              \
    {                                                                                   \
        pending = f_tile < n_tiles;                                                     \
        if (pending) {                                                                  \
            const unsigned char *from =                                                 \
                (brings_query ? a_base + (size_t)f_k0 * 2                               \
                              : reinterpret_cast<const unsigned char *>(a.base) +       \
                                    ((size_t)f_tile * BN * a.d + f_k0) * 2) + bring_off;\
            _Pragma("unroll") for (int i = 0; i < kInstrs; ++i)                         \
                bring_rows(from + (size_t)(kInstrRows * i) * a.d * 2 +                  \
                               16u * ((lane % kPieces) ^ PA_PLACE_MIX(kInstrRows * i + bring_row)), \
                           bring_to + (buf) * kStage + kInstrRows * i * kRow);          \
            f_k0 += kChunk;                                                             \
            if (f_k0 >= a.d) f_k0 = 0, f_tile += a.n_seg;                               \
        }                                                                               \
    }
// minus half the squared lengths of a tile's base rows, the columns of this
// wavefront (a column past the end: minus infinity, so it never passes)
#define PA_LOAD_NORMS(tile_)                                                            \
    _Pragma("unroll") for (int n = 0; n < WN; ++n) {                                    \
        const int64_t c = (tile_) * BN + (wc * WN + n) * 32 + col;                      \
        start[n] = c < a.n ? -0.5f * a.base_norm[c] : -INFINITY;                        \
    }
    float start[WN];
    if (seg < n_tiles) PA_LOAD_NORMS((int64_t)seg)
#pragma unroll
    for (int b = 0; b < kStages - 1; ++b) PA_FETCH_NEXT(b)
    if (pending) bring_wait<kAhead>(); else bring_wait<0>();
    __syncthreads();
    int buf = 0;

    for (int64_t tile = seg; tile < n_tiles; tile += a.n_seg) {
        floatx16 acc[WM][WN];
#pragma unroll
        for (int m = 0; m < WM; ++m)
#pragma unroll
            for (int n = 0; n < WN; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[m][n][r] = start[n];

#pragma unroll 1
        for (int k0 = 0; k0 < a.d; k0 += kChunk, buf = (buf + 1) % kStages) {
            // nobody reads the other buffer any more: the next chunk goes there
            PA_FETCH_NEXT((buf + kStages - 1) % kStages)
            // MFMA operands: lane l supplies eight consecutive elements of row
            // l % 32, the first or second eight of a group of 16 by l / 32 —
            // the same for both operands, which is all the sum needs
            const unsigned char *a_now = a_tile + buf * kStage, *b_now = b_tile + buf * kStage;
#pragma unroll
            for (int s = 0; s < kChunk / 16; ++s) {
                half8 av[WM], bv[WN];
                const unsigned at = swizzle ^ (32u * s);
#pragma unroll
                for (int m = 0; m < WM; ++m)
                    av[m] = *reinterpret_cast<const half8 *>(a_now + m * 32 * kRow + at);
#pragma unroll
                for (int n = 0; n < WN; ++n)
                    bv[n] = *reinterpret_cast<const half8 *>(b_now + n * 32 * kRow + at);
#pragma unroll
                for (int m = 0; m < WM; ++m)
#pragma unroll
                    for (int n = 0; n < WN; ++n)
                        acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            av[m], bv[n], acc[m][n], 0, 0, 0);
            }
            if (pending) bring_wait<kAhead>(); else bring_wait<0>();
            __syncthreads();
        }

        // the next tile's norms travel while this tile's sums are looked at
        if (tile + a.n_seg < n_tiles) PA_LOAD_NORMS(tile + a.n_seg)
        // a lane's 16 results of an instruction tile are
        // D[i = 8 * (r / 4) + 4 * (l / 32) + r % 4][j = l % 32]
        const int32_t c0 = (int32_t)(tile * BN) + wc * WN * 32 + col;
#pragma unroll
        for (int m = 0; m < WM; ++m) {
            // one row of instruction tiles at a time, so that its limits and
            // sums are all that is live
            __builtin_amdgcn_sched_barrier(0);
            const int row0 = (wr * WM + m) * 32 + 4 * half;
            float lim[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) lim[r] = limit[row0 + 8 * (r >> 2) + (r & 3)];
            if constexpr (SHORT) {
                unsigned live = 0;   // bit r: some lane's sum r is above its limit
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float best = acc[m][0][r];
#pragma unroll
                    for (int n = 1; n < WN; ++n) best = larger(best, acc[m][n][r]);
                    live |= __ballot(best > lim[r]) ? 1u << r : 0u;
                }
                if (!live) continue;
                // How many each of the 32 rows takes from this wavefront goes
                // to lane r + 16 half, and all their places are drawn with
                // one atomic instruction; then the entries are stored.
                int taken = 0;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    if ((live >> r) & 1) {
                        int low = 0, high = 0;
#pragma unroll
                        for (int n = 0; n < WN; ++n) {
                            const unsigned long long some = __ballot(acc[m][n][r] > lim[r]);
                            low += __popc((unsigned)some);
                            high += __popc((unsigned)(some >> 32));
                        }
                        taken = lane == r ? low : lane == 16 + r ? high : taken;
                    }
                }
                int place = 0;
                if (taken > 0)
                    place = atomicAdd(&count[(wr * WM + m) * 32 + 4 * (lane >> 4) +
                                             8 * ((lane & 15) >> 2) + (lane & 3)], taken);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    if ((live >> r) & 1) {
                        const int low = __builtin_amdgcn_readlane(place, r);
                        const int high = __builtin_amdgcn_readlane(place, 16 + r);
                        const unsigned row = row0 + 8 * (r >> 2) + (r & 3);
                        unsigned at = row * kCap + (half ? high : low);
#pragma unroll
                        for (int n = 0; n < WN; ++n) {
                            const bool in = acc[m][n][r] > lim[r];
                            const unsigned long long some = __ballot(in);
                            const unsigned mine = half ? (unsigned)(some >> 32) : (unsigned)some;
                            if (in) {
                                const unsigned to = at + __popc(mine & ((1u << col) - 1u));
                                my_score[to] = -2.f * acc[m][n][r];
                                my_id[to] = c0 + 32 * n;
                            }
                            at += __popc(mine);
                        }
                    }
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float best = acc[m][0][r];
                    if constexpr (WN == 4) {
                        best = larger(larger(best, acc[m][1][r], acc[m][2][r]), acc[m][3][r]);
                    } else {
#pragma unroll
                        for (int n = 1; n < WN; ++n) best = larger(best, acc[m][n][r]);
                    }
                    if (best > lim[r]) {  // rare after the first tiles
                        const int row = row0 + 8 * (r >> 2) + (r & 3);
#pragma unroll
                        for (int n = 0; n < WN; ++n) {
                            if (acc[m][n][r] > lim[r]) {
                                const unsigned at = row * kCap + atomicAdd(&count[row], 1);
                                my_score[at] = -2.f * acc[m][n][r];
                                my_id[at] = c0 + 32 * n;
                            }
                        }
                    }
                }
            }
        }
        __syncthreads();
        // every wavefront looks after kOwnRows lists: one that the next tile
        // could overflow is cut now
        {
            const int row = wave * kOwnRows + lane % kOwnRows;
            unsigned long long todo =
                __ballot(lane < kOwnRows && count[row] > KEEP + slack(KEEP));
            while (todo) {
                const int r = wave * kOwnRows + __builtin_ctzll(todo);
                todo &= todo - 1;
                const float b = cut_list<KEEP, BN>(my_score + (size_t)r * kCap,
                                                   my_id + (size_t)r * kCap, count[r], lane);
                if (lane == 0) count[r] = KEEP, limit[r] = -0.5f * b;
            }
        }
        // the next tile's first barrier comes before anything reads the
        // counts and limits again
    }
#undef PA_FETCH_NEXT
#undef PA_PLACE_MIX
#undef PA_LOAD_NORMS
    __syncthreads();
    {
        const int row = wave * kOwnRows + lane % kOwnRows;
        unsigned long long todo = __ballot(lane < kOwnRows && count[row] > KEEP);
        while (todo) {
            const int r = wave * kOwnRows + __builtin_ctzll(todo);
            todo &= todo - 1;
            cut_list<KEEP, BN>(my_score + (size_t)r * kCap, my_id + (size_t)r * kCap,
                               count[r], lane);
            if (lane == 0) count[r] = KEEP;
        }
    }
    __syncthreads();
    for (int r = t; r < BM; r += kThreads)
        if (q0 + r < a.m) a.cand_count[(size_t)seg * a.m + q0 + r] = count[r];
}

// The lists that the segments of a launch left for a row become one, in the
// place of the first segment's: the `KEEP` smallest of them all.  A wavefront
// per row; what is below the limit so far is appended and the list cut when it
// is nearly full, as in knn_kernel: a handful of cuts for sixteen segments, where
// a cut after every segment made fifteen (2048 rows 124 us).
constexpr int kRankWaves = 4;
constexpr int kMaxRankDim = 2048;   // rows of a workgroup and their lists fit 64 KB of LDS

template <int KEEP>
__global__ __launch_bounds__(kWave * kRankWaves) void merge_kernel(
    float *__restrict__ score, int32_t *__restrict__ id, int32_t *__restrict__ count,
    int64_t m, int n_seg) {
    constexpr int kCap = KEEP + slack(KEEP) + kMaxBN;
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t row = (int64_t)blockIdx.x * kRankWaves + threadIdx.x / kWave;
    if (row >= m) return;
    float *my_score = score + (size_t)row * kCap;
    int32_t *my_id = id + (size_t)row * kCap;
    int n = uni(count[row]);
    float limit = INFINITY;
    // the wavefront's stores before its other lanes' loads of the list, and
    // those before the next stores
    auto settle = []() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    };
    auto cut = [&]() {
        settle();
        limit = uni(cut_list<KEEP, kMaxBN>(my_score, my_id, n, lane));
        n = KEEP;
        settle();
    };
    for (int seg = 1; seg < n_seg; ++seg) {
        const size_t at = (size_t)seg * m + row;
        const int cnt = uni(count[at]);
        // up to 256 entries of the segment's list in one trip (64 at a time, and their
        // ids behind the comparison: 1024 rows of 4 lists 36 us, now 25; 8192 of 8
        // lists 104, now 74)
        constexpr int kAtOnce = KEEP < 256 ? KEEP / kWave : 4;
        for (int base = 0; base < cnt; base += kAtOnce * kWave) {
            float x[kAtOnce];
            int32_t node[kAtOnce];
#pragma unroll
            for (int r = 0; r < kAtOnce; ++r) {
                const int i = base + r * kWave + lane;
                x[r] = i < cnt ? score[at * kCap + i] : INFINITY;
                node[r] = i < cnt ? id[at * kCap + i] : -1;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < kAtOnce; ++r) {
                const bool in = base + r * kWave + lane < cnt && x[r] < limit;
                const unsigned long long mask = __ballot(in);
                if (in) {
                    my_score[n + lane_rank(mask)] = x[r];
                    my_id[n + lane_rank(mask)] = node[r];
                }
                n += __popcll(mask);
                if (n > kCap - kWave) cut();
            }
        }
    }
    if (n > KEEP) cut();
    if (lane == 0) count[row] = n;
}

// The exact squared distance between a row in LDS (`mine`) and row `row`, the
// float arithmetic of the search itself (differences, then squares, summed),
// by the 16 lanes of a team, `place` the lane's place in it, every lane 16
// bytes of the row per step.  Every lane of the wavefront calls this.
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float team_square_dist(const floatx4 *mine, const floatx4 *row, int d4,
                                                  int place, bool ok) {
    float sum = 0.f;
    if (ok) {
        for (int i = place; i < d4; i += 16) {
            const floatx4 x = row[i], y = mine[i];
            const float e0 = x[0] - y[0], e1 = x[1] - y[1], e2 = x[2] - y[2], e3 = x[3] - y[3];
            sum = fmaf(e0, e0, sum);
            sum = fmaf(e1, e1, sum);
            sum = fmaf(e2, e2, sum);
            sum = fmaf(e3, e3, sum);
        }
    }
#pragma unroll
    for (int step = 8; step >= 1; step >>= 1) sum += __shfl_xor(sum, step, 16);
    return sum;
}

// The same for two rows, whose loads are in flight together.
__device__ __forceinline__ void team_square_dists(const floatx4 *mine, const floatx4 *row0,
                                                  const floatx4 *row1, int d4, int place,
                                                  float &sum0, float &sum1) {
    sum0 = sum1 = 0.f;
    for (int i = place; i < d4; i += 16) {
        const floatx4 x = row0[i], z = row1[i], y = mine[i];
        const float e0 = x[0] - y[0], e1 = x[1] - y[1], e2 = x[2] - y[2], e3 = x[3] - y[3];
        const float f0 = z[0] - y[0], f1 = z[1] - y[1], f2 = z[2] - y[2], f3 = z[3] - y[3];
        sum0 = fmaf(e0, e0, sum0), sum1 = fmaf(f0, f0, sum1);
        sum0 = fmaf(e1, e1, sum0), sum1 = fmaf(f1, f1, sum1);
        sum0 = fmaf(e2, e2, sum0), sum1 = fmaf(f2, f2, sum1);
        sum0 = fmaf(e3, e3, sum0), sum1 = fmaf(f3, f3, sum1);
    }
#pragma unroll
    for (int step = 8; step >= 1; step >>= 1) {
        sum0 += __shfl_xor(sum0, step, 16);
        sum1 += __shfl_xor(sum1, step, 16);
    }
}

// Exact squared distances from query row first + q to its candidates.  A
// wavefront per query, its row in LDS; 16 lanes per candidate, four candidates
// at a time.  A candidate that is -1, out of range or the query row itself gets
// infinity.
__global__ __launch_bounds__(kWave * kRankWaves) void rerank_kernel(
    const float *__restrict__ rows, const int64_t *__restrict__ cand,
    float *__restrict__ out, int64_t m, int64_t first, int64_t n, int d, int k) {
    extern __shared__ __align__(16) unsigned char rank_lds[];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int64_t q = (int64_t)blockIdx.x * kRankWaves + wave;
    const int d4 = d / 4;
    floatx4 *mine = reinterpret_cast<floatx4 *>(rank_lds) + wave * d4;
    if (q < m) {
        const floatx4 *src = reinterpret_cast<const floatx4 *>(rows + (size_t)(first + q) * d);
        for (int i = lane; i < d4; i += kWave) mine[i] = src[i];
    }
    __syncthreads();
    if (q >= m) return;
    const int team = lane >> 4, place = lane & 15;
    for (int j0 = 0; j0 < k; j0 += 4) {
        const int j = j0 + team;
        const int64_t id = j < k ? cand[(size_t)q * k + j] : -1;
        const bool ok = id >= 0 && id < n && id != first + q;
        const float sum = team_square_dist(
            mine, reinterpret_cast<const floatx4 *>(rows + (ok ? (size_t)id * d : 0)), d4, place, ok);
        if (place == 0 && j < k) out[(size_t)q * k + j] = ok ? sum : INFINITY;
    }
}

// The ranking that follows knn_kernel in one pass: the distances of a row's
// list, as rerank_kernel makes them, sorted in LDS, the k closest written out;
// equal distances in the order of the half-precision scores where lists were
// merged, and then in that of the rows: a candidate's place in its list is
// where knn_kernel's wavefronts happened to put it, and two runs over the same
// rows with equal ones among them would name them in different orders.  What
// bounds it is the gathering of the candidates' rows; the sort of 256 entries
// (36 passes of two exchanges a lane) hides behind other wavefronts' reads,
// where ranking in steps of torch (ids widened, top-k, gather, masks) wrote and
// read the table several times.
template <int KEEP, bool TWO>
__global__ __launch_bounds__(kWave * kRankWaves) void rank_kernel(
    const float *__restrict__ rows, const float *__restrict__ cand_score,
    const int32_t *__restrict__ cand_id, const int32_t *__restrict__ count,
    int64_t *__restrict__ out_id, float *__restrict__ out_dist, int64_t m, int64_t first,
    int64_t n, int d, int k, int hide_inf, int merged) {
    constexpr int kCap = KEEP + slack(KEEP) + kMaxBN;
    constexpr unsigned kPlaces = 511;   // the bits of an entry that are its place in the list
    extern __shared__ __align__(16) unsigned char rank_lds[];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int64_t q = (int64_t)blockIdx.x * kRankWaves + wave;
    const int d4 = d / 4;
    // per wavefront: (distance, 23 bits of the score, place in the list) of the
    // candidates, and the row
    unsigned long long *entry =
        reinterpret_cast<unsigned long long *>(rank_lds) + wave * KEEP;
    floatx4 *mine = reinterpret_cast<floatx4 *>(rank_lds + kRankWaves * KEEP * 8) + wave * d4;
    if (q >= m) return;
    const floatx4 *src = reinterpret_cast<const floatx4 *>(rows + (size_t)(first + q) * d);
    for (int i = lane; i < d4; i += kWave) mine[i] = src[i];
    const int32_t *ids = cand_id + (size_t)q * kCap;
    const int cnt = min(KEEP, uni(count[q]));
    // the list, an id a lane and 64 of them a register; what an entry holds below
    // its distance
    int32_t held[KEEP / kWave];
#pragma unroll
    for (int r = 0; r < KEEP / kWave; ++r) {
        const int j = r * kWave + lane;
        held[r] = j < cnt ? ids[j] : -1;
        const unsigned score =
            merged && j < cnt ? ordered(cand_score[(size_t)q * kCap + j]) : 0u;
        entry[j] = j < cnt ? (score & ~kPlaces) | (unsigned)j : ~0ull;
    }
    wave_sync();
    const int team = lane >> 4, place = lane & 15;
    unsigned *high = reinterpret_cast<unsigned *>(entry) + 1;
#pragma unroll
    for (int r = 0; r < KEEP / kWave; ++r) {
        const int here = min(kWave, cnt - r * kWave);
        for (int j0 = 0; !TWO && j0 < here; j0 += 4) {
            const int at = r * kWave + j0 + team;
            const int32_t id = __shfl(held[r], j0 + team);
            const bool ok = id >= 0 && id < n && id != first + q;
            const float sum = team_square_dist(
                mine, reinterpret_cast<const floatx4 *>(rows + (ok ? (size_t)id * d : 0)), d4,
                place, ok);
            if (place == 0 && at < cnt) high[2 * at] = __float_as_uint(ok ? sum : INFINITY);
        }
#pragma unroll 1
        for (int j0 = 0; TWO && j0 < here; j0 += 8) {
            // two candidates a team, their rows requested together
            const int j = j0 + team;
            const int32_t id0 = __shfl(held[r], j), id1 = __shfl(held[r], j + 4);
            const bool ok0 = id0 >= 0 && id0 < n && id0 != first + q;
            const bool ok1 = id1 >= 0 && id1 < n && id1 != first + q;
            const floatx4 *row0 =
                reinterpret_cast<const floatx4 *>(rows + (ok0 ? (size_t)id0 * d : 0));
            const floatx4 *row1 =
                reinterpret_cast<const floatx4 *>(rows + (ok1 ? (size_t)id1 * d : 0));
            float sum0, sum1;
            team_square_dists(mine, row0, row1, d4, place, sum0, sum1);
            if (place == 0) {
                const int at = r * kWave + j;
                if (at < cnt) high[2 * at] = __float_as_uint(ok0 ? sum0 : INFINITY);
                if (at + 4 < cnt) high[2 * at + 8] = __float_as_uint(ok1 ? sum1 : INFINITY);
            }
        }
    }
    wave_sync();
#pragma unroll 1
    for (int size = 2; size <= KEEP; size <<= 1) {
#pragma unroll 1
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
#pragma unroll
            for (int t0 = 0; t0 < KEEP / 2; t0 += kWave) {
                const int t = t0 + lane;
                const int i = ((t & ~(stride - 1)) << 1) | (t & (stride - 1));
                if (KEEP / 2 >= kWave || t < KEEP / 2) {
                    const unsigned long long x = entry[i], y = entry[i | stride];
                    bool after = x > y;
                    if (x != y && (x ^ y) <= kPlaces && x != ~0ull && y != ~0ull)
                        after = ids[x & kPlaces] > ids[y & kPlaces];
                    if (after == ((i & size) == 0) && x != y) entry[i] = y, entry[i | stride] = x;
                }
            }
            wave_sync();
        }
    }
    for (int i = lane; i < k; i += kWave) {
        const unsigned long long e = entry[i];
        const bool none = (unsigned)(e >> 32) == 0xffffffffu;
        const int32_t id = none ? -1 : ids[(unsigned)e & kPlaces];
        const float dist = none ? INFINITY : __uint_as_float((unsigned)(e >> 32));
        out_id[(size_t)q * k + i] = hide_inf && isinf(dist) ? -1 : (int64_t)id;
        out_dist[(size_t)q * k + i] = dist;
    }
}

// Nodes or rows of a launch of the kernels with a wavefront or a workgroup for
// each: a launch holds fewer than 2^32 work-items, and 2^22 workgroups of 256
// are 2^30.
constexpr int64_t kLaunchNodes = 1ll << 22;

// What half precision leaves of the rows: x = row * scale, clamped to the half
// range, lo = half(x - half(x)), padded with zeros to d_pad elements and n_pad
// rows.  A wavefront per row, four elements a lane and step, one pass over the
// rows where the same steps as tensor operations made six.
typedef _Float16 half4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(kWave * kRankWaves) void low_kernel(
    const float *__restrict__ rows, _Float16 *__restrict__ lo, int64_t first, int64_t n,
    int64_t n_pad, int d, int d_pad, float scale, float most) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t row = first + (int64_t)blockIdx.x * kRankWaves + threadIdx.x / kWave;
    if (row >= n_pad) return;
    const float *src = rows + (size_t)row * d;
    for (int i = 4 * lane; i < d_pad; i += 4 * kWave) {
        half4 l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float x = row < n && i + e < d ? src[i + e] * scale : 0.f;
            x = x > most ? most : x < -most ? -most : x;   // NaN stays
            l[e] = (_Float16)(x - (float)(_Float16)x);
        }
        *reinterpret_cast<half4 *>(lo + (size_t)row * d_pad + i) = l;
    }
}

// One step of a walk along the edges of adj [n, deg] (negative: no edge) over
// marks of one byte a node.  Forward: 1 is a node just reached, whose neighbours
// are reached now (it becomes 2); backward: a node with a marked neighbour is
// marked (2; 1 is a node the walk starts from, whose row is only looked at for
// its numbers).  A node may be reached and go on within one launch, and one
// that two wavefronts reach at a time may be gone over twice: the marks only
// grow, and a step that changes nothing (bit 0 of `status` stays 0 in the
// `last` one) is the end.  A number that is no node's is no edge and sets bit
// 1.  A wavefront per node; most nodes are one byte read.
__global__ __launch_bounds__(256) void reach_kernel(
    const int64_t *__restrict__ adj, unsigned char *mark, int *status, int64_t first, int64_t n,
    int deg, int backward, int last) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t node =
        first + (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (node >= n) return;
    const int state = mark[node];
    if (backward ? state == 2 : state != 1) return;
    if (state == 1 && lane == 0) mark[node] = 2;
    bool found = false, beyond = false;
    for (int e = lane; e < deg; e += kWave) {
        const int64_t v = adj[(size_t)node * deg + e];
        beyond |= v >= n;
        if (v < 0 || v >= n) continue;
        if (backward) {
            found |= mark[v] != 0;
        } else if (mark[v] == 0) {
            mark[v] = 1;
            found = true;
        }
    }
    const bool grown = __ballot(found) && !(backward && state == 1);
    const int bits = (__ballot(beyond) ? 2 : 0) | (grown && last ? 1 : 0);
    if (lane != 0) return;
    if (backward && grown) mark[node] = 2;
    // one wavefront's word is enough: most find the bit set
    if (bits & ~__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicOr(status, bits);
}

__global__ void clear_flag(int *flag) { *flag = 0; }

// Occlusion pruning of a node's candidate list (closest first): candidate j
// is kept unless a candidate kept before it is closer to it than the node
// itself is, until m_keep are kept; with `fill` the closest rejected ones top
// the row up to m_keep.  One wavefront per node; the kept set is a bit mask
// that every lane carries, a step tests one row of the node's table of
// candidate-to-candidate distances against it.
__global__ __launch_bounds__(256) void prune_kernel(
    const float *__restrict__ pair, const float *__restrict__ cand_dist,
    int32_t *__restrict__ selected, int64_t n, int k, int m_keep, int fill) {
    constexpr int kWords = 8;  // k <= 512
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t node = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (node >= n) return;
    const float *table = pair + (size_t)node * k * k;
    const float *dist = cand_dist + (size_t)node * k;
    int32_t *out = selected + (size_t)node * m_keep;
    unsigned long long kept[kWords];
#pragma unroll
    for (int w = 0; w < kWords; ++w) kept[w] = 0;
    int count = 0;
    for (int j = 0; j < k && count < m_keep; ++j) {
        const float own = dist[j];
        bool hit = false;
        // only candidates before j can have been kept
#pragma unroll
        for (int w = 0; w < kWords; ++w) {
            const int r = 64 * w + lane;
            if (64 * w < j && r < j && ((kept[w] >> lane) & 1ull))
                hit |= table[(size_t)j * k + r] < own;
        }
        if (!__ballot(hit)) {
#pragma unroll
            for (int w = 0; w < kWords; ++w)
                if (j >> 6 == w) kept[w] |= 1ull << (j & 63);
            if (lane == 0) out[count] = j;
            count += 1;
        }
    }
    if (fill) {
        for (int j = 0; j < k && count < m_keep; ++j) {
            bool is_kept = false;
#pragma unroll
            for (int w = 0; w < kWords; ++w)
                if (j >> 6 == w) is_kept = (kept[w] >> (j & 63)) & 1ull;
            if (is_kept) continue;
            if (lane == 0) out[count] = j;
            count += 1;
        }
    }
    for (int i = count + lane; i < m_keep; i += kWave) out[i] = -1;
}

// Occlusion pruning straight from the rows: the same rule as prune_kernel,
// with the candidate-to-candidate distances made on the spot.  Only a kept
// candidate can block another one, and few are kept (a dozen or two of 240), so
// the candidates are taken 64 at a time, closest first, and a block's rows are
// multiplied with themselves (the lower triangle) and with the rows kept
// before them: two fifths of the products of all pairs, and the blocks after
// the m_keep-th kept candidate are never looked at.
//
// A workgroup of four wavefronts takes one node.  It gathers rows chunk by
// chunk into LDS (the transfers of knn_kernel, every lane with the address of
// its own row) and multiplies them on the matrix cores — rows as two
// half-precision parts, x = hi + lo, and hi.hi + hi.lo + lo.hi for the product,
// which is the float product to about 22 bits.  |a|^2 + |b|^2 - 2 a.b <
// dist(node, a) is one bit per pair, and the first wavefront walks a block's
// candidates from one that is kept to the next.  What bounds it is the
// gathering of rows; one staging buffer, so that four workgroups share a
// compute unit and each one's waits and serial walk hide behind the others'.
// 120 000 nodes of 240 candidates of 768 floats, 48 to keep: 34.8 -> 15.0 ms
// against all pairs on eight wavefronts with a double buffer, one workgroup
// per compute unit; 20 011 nodes of 96 floats, 16 to keep: 2.67 -> 0.38 ms.
struct PruneRowsArgs {
    const _Float16 *hi, *lo;
    const float *norm;        // squared lengths of the scaled rows
    const int64_t *cand;      // [n, k] row numbers, closest first, -1 after the last
    const float *cand_dist;   // [n, k] squared distances to the node, unscaled
    int32_t *selected;        // [n, m_keep]
    int64_t n, first;         // this launch takes nodes first .. first + gridDim.x
    int64_t n_rows;           // rows behind hi / lo / norm: a candidate at or beyond is no candidate
    int d, k, m_keep, fill;
    float scale2;             // (scaled / unscaled) squared
};

__global__ __launch_bounds__(256, 4) void prune_rows_kernel(PruneRowsArgs a) {
    constexpr int kMaxCand = 256;
    constexpr int kBlock = 64;                 // candidates looked at together
    constexpr int kSide = 32;                  // kept candidates multiplied with them at a time
    constexpr int kRows = kBlock + kSide;      // rows staged
    constexpr int kRow = kChunk * 2;           // bytes of a staged row
    constexpr int kPart = kRows * kRow;        // one part (hi or lo) of a chunk
    __shared__ __align__(1024) unsigned char stage[2 * kPart];
    __shared__ int64_t row_of[kMaxCand];       // candidate -> row
    __shared__ float len2[kMaxCand], reach[kMaxCand];
    __shared__ unsigned self_bits[kBlock][2];  // bit b of [a]: b of the block would block a of it
    __shared__ unsigned side_bits[kBlock];     // not 0: a kept one of this pass blocks a
    __shared__ int kept_at[kMaxCand];          // the candidates kept, in order
    __shared__ int valid_count, kept_count;
    const int t = threadIdx.x;
    const int lane = t & (kWave - 1), wave = uni(t / kWave);
    const int col = lane & 31, half = lane >> 5;
    const int64_t node = a.first + blockIdx.x;
    const int64_t *ids = a.cand + (size_t)node * a.k;

    // the candidates' rows, lengths and distances.  A candidate is a row
    // number inside the set; what is none (what lies behind the list, too)
    // repeats the first candidate's row and can be blocked by nothing
    if (t == 0) valid_count = 0;
    __syncthreads();
    {
        auto cand_at = [&](int i) -> int64_t {
            const int64_t id = i < a.k ? ids[i] : -1;
            return id < a.n_rows ? id : -1;
        };
        const int64_t first_id = cand_at(0);
        const int64_t id = cand_at(t);
        row_of[t] = id >= 0 ? id : first_id >= 0 ? first_id : 0;
        len2[t] = id >= 0 ? a.norm[id] : 0.f;
        reach[t] = id >= 0 ? a.cand_dist[(size_t)node * a.k + t] * a.scale2 : -INFINITY;
        const unsigned long long valid = __ballot(id >= 0);
        if (lane == 0) atomicAdd(&valid_count, (int)__popcll(valid));
    }
    __syncthreads();
    const int k_valid = uni(valid_count);

    // transfers: an instruction brings 8 rows, lane l the piece that belongs
    // at place l % 8 of row l / 8 (places as in knn_kernel); wavefront w brings
    // rows 24 w .. 24 w + 23 of both parts
    constexpr int kBrings = kRows / 8 / 4;
    const int bring_row = lane >> 3;
    const unsigned char *hi = reinterpret_cast<const unsigned char *>(a.hi);
    const unsigned char *lo = reinterpret_cast<const unsigned char *>(a.lo);
    const unsigned bring_to =
        (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)stage;
    const unsigned mix = (col >> 1) & 7;
    const unsigned swizzle = 16u * (half ^ (mix & 1)) + 32u * (mix >> 1);
    // wavefront w multiplies rows 32 (w % 2) .. + 31 of the block: the first
    // two with the block itself, the other two with the kept rows
    const int m0 = 32 * (wave & 1);
    const bool with_side = wave >= 2;

    int count = 0;
    int32_t *out = a.selected + (size_t)node * a.m_keep;
    unsigned long long kept_mask[kMaxCand / kBlock];   // for the filling
#pragma unroll
    for (int blk = 0; blk < kMaxCand / kBlock; ++blk) {
        kept_mask[blk] = 0;
        const int c0 = blk * kBlock;
        if (c0 >= k_valid || count >= a.m_keep) continue;
        unsigned long long blocked = 0;   // of the block's candidates, in the first wavefront
        // passes over the kept ones, 32 a time; the first pass does the block itself
        int side0 = 0;
        do {
            const int n_side = min(kSide, count - side0);   // <= 0: none yet
            const bool self_pass = side0 == 0;
            size_t from[kBrings];
            bool wanted[kBrings];
#pragma unroll
            for (int i = 0; i < kBrings; ++i) {
                const int r8 = (wave * kBrings + i) * 8;
                wanted[i] = r8 < kBlock || r8 - kBlock < n_side;
                const int r = r8 + bring_row;
                int c = 0;
                if (r < kBlock) c = c0 + r;
                else if (r - kBlock < n_side) c = kept_at[side0 + r - kBlock];
                from[i] = (size_t)row_of[c] * a.d * 2 + 16u * ((lane & 7) ^ ((r >> 1) & 7));
            }
            floatx16 acc[2];
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
            // tiles of this wavefront: the block's columns 0 .. m0 + 31, or
            // the kept rows
            const int n_tiles = with_side ? (n_side > 0 ? 1 : 0) : self_pass ? 1 + (wave & 1) : 0;
            const unsigned char *a_tile = stage + (m0 + col) * kRow;
            const unsigned char *b_tile = stage + ((with_side ? kBlock : 0) + col) * kRow;
#pragma unroll 1
            for (int k0 = 0; k0 < a.d; k0 += kChunk) {
#pragma unroll
                for (int i = 0; i < kBrings; ++i) {
                    if (wanted[i]) {
                        const unsigned to = bring_to + (wave * kBrings + i) * 8 * kRow;
                        bring_rows(hi + from[i] + (size_t)k0 * 2, to);
                        bring_rows(lo + from[i] + (size_t)k0 * 2, to + kPart);
                    }
                }
                bring_wait<0>();
                __syncthreads();
                if (n_tiles > 0) {
#pragma unroll
                    for (int s = 0; s < kChunk / 16; ++s) {
                        const unsigned at = swizzle ^ (32u * s);
                        const half8 ah = *reinterpret_cast<const half8 *>(a_tile + at);
                        const half8 al = *reinterpret_cast<const half8 *>(a_tile + kPart + at);
                        const half8 bh = *reinterpret_cast<const half8 *>(b_tile + at);
                        const half8 bl = *reinterpret_cast<const half8 *>(b_tile + kPart + at);
                        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, acc[0], 0, 0, 0);
                        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, acc[0], 0, 0, 0);
                        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, acc[0], 0, 0, 0);
                        if (n_tiles > 1) {
                            const half8 ch = *reinterpret_cast<const half8 *>(b_tile + 32 * kRow + at);
                            const half8 cl = *reinterpret_cast<const half8 *>(b_tile + 32 * kRow + kPart + at);
                            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, ch, acc[1], 0, 0, 0);
                            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, cl, acc[1], 0, 0, 0);
                            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, ch, acc[1], 0, 0, 0);
                        }
                    }
                }
                __syncthreads();
            }

            // a lane's 16 results of an instruction tile are
            // D[i = 8 * (r / 4) + 4 * (l / 32) + r % 4][j = l % 32]: one ballot
            // is the word of 32 columns for two rows
            auto tile_bits = [&](const floatx16 &sums, float len_b, bool real, unsigned *to,
                                 int pitch) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = m0 + 8 * (r >> 2) + 4 * half + (r & 3);
                    const float pair = (len2[c0 + row] + len_b) - 2.f * sums[r];
                    const unsigned long long word = __ballot(real && pair < reach[c0 + row]);
                    if (col == 0)
                        to[row * pitch] = half ? (unsigned)(word >> 32) : (unsigned)word;
                }
            };
            if (with_side) {
                if (n_tiles > 0) {
                    const bool real = col < n_side;
                    tile_bits(acc[0], real ? len2[kept_at[side0 + col]] : 0.f, real,
                              side_bits, 1);
                }
            } else if (n_tiles > 0) {
                tile_bits(acc[0], len2[c0 + col], true, &self_bits[0][0], 2);
                if (n_tiles > 1) tile_bits(acc[1], len2[c0 + 32 + col], true, &self_bits[0][1], 2);
            }
            __syncthreads();
            if (wave == 0 && n_side > 0) blocked |= __ballot(side_bits[lane] != 0);
            side0 += kSide;
        } while (side0 < count);

        // the walk: lane l holds the bits of the block's candidate l, of which
        // those of candidates before it count
        if (wave == 0) {
            const unsigned b0 = self_bits[lane][0], b1 = lane >= 32 ? self_bits[lane][1] : 0u;
            const unsigned long long mine = ((unsigned long long)b1 << 32) | b0;
            unsigned long long alive = ~blocked;
            if (k_valid - c0 < kBlock) alive &= (1ull << (k_valid - c0)) - 1;
            unsigned long long kept = 0;
            int n = count;
            while (alive && n < a.m_keep) {
                const int j = __builtin_ctzll(alive);
                kept |= 1ull << j;
                alive &= ~1ull << j;                          // those after it
                alive &= ~__ballot((mine >> j) & 1ull);       // that it does not block
                n += 1;
            }
            if ((kept >> lane) & 1ull) {
                const int place = count + lane_rank(kept);
                kept_at[place] = c0 + lane;
                out[place] = c0 + lane;
            }
            kept_mask[blk] = kept;
            if (lane == 0) kept_count = n;
        }
        __syncthreads();
        count = uni(kept_count);
    }
    if (wave != 0) return;
    // the closest rejected ones
    if (a.fill) {
#pragma unroll
        for (int blk = 0; blk < kMaxCand / kBlock; ++blk) {
            const int c = blk * kBlock + lane;
            const bool rejected = c < k_valid && !((kept_mask[blk] >> lane) & 1ull);
            const unsigned long long mask = __ballot(rejected);
            const int place = count + lane_rank(mask);
            if (rejected && place < a.m_keep) out[place] = c;
            count += __popcll(mask);
        }
    }
    for (int i = count + lane; i < a.m_keep; i += kWave) out[i] = -1;
}

// The form in use: 2 x 4 wavefronts of 4 x 2 instruction tiles, 256 query rows
// against 256 base rows per tile; one workgroup per compute unit (150 KB of
// LDS, 256 registers a lane).
constexpr int kWR = 2, kWC = 4, kWM = 4, kWN = 2;
constexpr int kBM = 32 * kWR * kWM;

constexpr int kShortWalk = 32;   // tiles

template <int KEEP>
int launch_knn(const KnnArgs &a, hipStream_t stream) {
    constexpr int kBN = 32 * kWC * kWN;
    const dim3 grid((unsigned)((a.m + kBM - 1) / kBM), (unsigned)a.n_seg);
    const int64_t tiles = (a.n + kBN - 1) / kBN;   // dealt to the segments
    if ((tiles + a.n_seg - 1) / a.n_seg <= kShortWalk)
        knn_kernel<KEEP, true, kWR, kWC, kWM, kWN><<<grid, 64 * kWR * kWC, 0, stream>>>(a);
    else
        knn_kernel<KEEP, false, kWR, kWC, kWM, kWN><<<grid, 64 * kWR * kWC, 0, stream>>>(a);
    return (int)hipGetLastError();
}

}  // namespace

extern "C" int64_t pa_knn_list_capacity(int keep) {
    return keep == 64 || keep == 128 || keep == 256 || keep == 512 ? keep + slack(keep) + kMaxBN : 0;
}

extern "C" int pa_knn_tile_rows(void) { return kRowPad; }

extern "C" int pa_knn(float *cand_score, int32_t *cand_id, int32_t *cand_count,
                      const void *query_f16, const void *base_f16,
                      const float *base_norm, int64_t m, int64_t n, int d,
                      int keep, int n_seg, void *stream_) {
    if (m < 0 || n < 0 || n_seg < 1 || n_seg > 65535) return PA_E_SHAPE;
    // ids are 32 bits, and a launch holds fewer than 2^32 work-items
    if (n >= (1ll << 31) || (m + kBM - 1) / kBM * n_seg >= (1ll << 32) / (64 * kWR * kWC))
        return PA_E_RANGE;
    if (d <= 0 || d % kChunk) return PA_E_DIM;
    if (keep != 64 && keep != 128 && keep != 256 && keep != 512) return PA_E_SHAPE;
    if (m == 0) return PA_OK;
    if (n == 0) return PA_E_SHAPE;
    if (!cand_score || !cand_id || !cand_count || !query_f16 || !base_f16 || !base_norm)
        return PA_E_NULL;
    KnnArgs a;
    a.query = reinterpret_cast<const _Float16 *>(query_f16);
    a.base = reinterpret_cast<const _Float16 *>(base_f16);
    a.base_norm = base_norm;
    a.cand_score = cand_score, a.cand_id = cand_id, a.cand_count = cand_count;
    a.m = m, a.n = n, a.d = d, a.n_seg = n_seg;
    hipStream_t stream = (hipStream_t)stream_;
    switch (keep) {
        case 64: return launch_knn<64>(a, stream);
        case 128: return launch_knn<128>(a, stream);
        case 256: return launch_knn<256>(a, stream);
        default: return launch_knn<512>(a, stream);
    }
}

extern "C" int pa_knn_rerank(float *dist, const float *rows, const int64_t *cand,
                             int64_t m, int64_t first, int64_t n, int d, int k,
                             void *stream_) {
    if (m < 0 || n < 0 || first < 0 || first + m > n || k < 1) return PA_E_SHAPE;
    if (d <= 0 || d % 4 || d > 4096) return PA_E_DIM;
    if (m >= (1ll << 32) / kWave) return PA_E_RANGE;   // work-items of the launch
    if (m == 0) return PA_OK;
    if (!dist || !rows || !cand) return PA_E_NULL;
    const unsigned lds = (unsigned)(kRankWaves * d * sizeof(float));
    rerank_kernel<<<(unsigned)((m + kRankWaves - 1) / kRankWaves), kWave * kRankWaves, lds,
                    (hipStream_t)stream_>>>(rows, cand, dist, m, first, n, d, k);
    return (int)hipGetLastError();
}

extern "C" int pa_knn_rank(int64_t *out_id, float *out_dist, float *cand_score,
                           int32_t *cand_id, int32_t *cand_count, const float *rows, int64_t m,
                           int64_t first, int64_t n, int d, int keep, int n_seg, int k,
                           int hide_inf, void *stream_) {
    if (m < 0 || n < 0 || first < 0 || first + m > n || n_seg < 1) return PA_E_SHAPE;
    if (keep != 64 && keep != 128 && keep != 256 && keep != 512) return PA_E_SHAPE;
    if (k < 1 || k > keep) return PA_E_SHAPE;
    if (d <= 0 || d % 4 || d > kMaxRankDim) return PA_E_DIM;
    // row numbers are 32 bits; work-items of a launch
    if (n >= (1ll << 31) || m >= (1ll << 32) / kWave) return PA_E_RANGE;
    if (m == 0) return PA_OK;
    if (!out_id || !out_dist || !cand_score || !cand_id || !cand_count || !rows) return PA_E_NULL;
    hipStream_t stream = (hipStream_t)stream_;
    const unsigned blocks = (unsigned)((m + kRankWaves - 1) / kRankWaves);
    const unsigned lds = (unsigned)(kRankWaves * (d * sizeof(float) + keep * 8));
    // Two candidates a team at a time where few rows are ranked, which is a chain of
    // trips to memory, or rows are short; else one, whose rows stay in L2.  Kernel
    // alone, one / two, us, 96 floats: 1024 rows 62 / 42, 8192 123 / 84; 768 floats: 1024
    // 178 / 118, 4096 296 / 189, 8192 378 / 485, 54 464 4855 / 5473; builds of 150 000
    // x 256 37.7 (one from 8192 rows on) / 38.5 ms.
    const bool two = m <= 4096 || d <= 128;
#define PA_RANK(KEEP_)                                                                        \
    {                                                                                         \
        if (n_seg > 1)                                                                        \
            merge_kernel<KEEP_><<<blocks, kWave * kRankWaves, 0, stream>>>(                   \
                cand_score, cand_id, cand_count, m, n_seg);                                   \
        (two ? rank_kernel<KEEP_, true> : rank_kernel<KEEP_, false>)                          \
            <<<blocks, kWave * kRankWaves, lds, stream>>>(rows, cand_score, cand_id,          \
                                                          cand_count, out_id, out_dist, m,    \
                                                          first, n, d, k, hide_inf,           \
                                                          n_seg > 1);                         \
    }
    switch (keep) {
        case 64: PA_RANK(64) break;
        case 128: PA_RANK(128) break;
        case 256: PA_RANK(256) break;
        default: PA_RANK(512) break;
    }
#undef PA_RANK
    return (int)hipGetLastError();
}

extern "C" int pa_rows_low(void *lo_f16, const float *rows, int64_t n, int64_t n_pad, int d,
                           int d_pad, float scale, float most, void *stream_) {
    if (n < 0 || n_pad < n) return PA_E_SHAPE;
    if (d <= 0 || d_pad < d || d_pad % 4) return PA_E_DIM;
    if (n_pad == 0) return PA_OK;
    if ((n > 0 && !rows) || !lo_f16) return PA_E_NULL;
    for (int64_t first = 0; first < n_pad; first += kLaunchNodes) {
        const int64_t count = n_pad - first < kLaunchNodes ? n_pad - first : kLaunchNodes;
        low_kernel<<<(unsigned)((count + kRankWaves - 1) / kRankWaves), kWave * kRankWaves, 0,
                     (hipStream_t)stream_>>>(rows, reinterpret_cast<_Float16 *>(lo_f16), first, n,
                                             n_pad, d, d_pad, scale, most);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return (int)err;
    }
    return PA_OK;
}

extern "C" int pa_graph_reach(unsigned char *mark, int *status, const int64_t *adj, int64_t n,
                              int deg, int backward, int steps, void *stream_) {
    if (n < 0 || deg < 1 || steps < 1) return PA_E_SHAPE;
    if (n == 0) return PA_OK;
    if (!mark || !status || !adj) return PA_E_NULL;
    hipStream_t stream = (hipStream_t)stream_;
    clear_flag<<<1, 1, 0, stream>>>(status);
    for (int step = 0; step < steps; ++step) {
        for (int64_t first = 0; first < n; first += kLaunchNodes) {
            const int64_t count = n - first < kLaunchNodes ? n - first : kLaunchNodes;
            reach_kernel<<<(unsigned)((count + 3) / 4), 256, 0, stream>>>(
                adj, mark, status, first, n, deg, backward, step + 1 == steps);
        }
    }
    return (int)hipGetLastError();
}

extern "C" int pa_graph_prune_rows(int32_t *selected, const void *rows_hi_f16,
                                   const void *rows_lo_f16, const float *norm,
                                   const int64_t *cand, const float *cand_dist,
                                   int64_t n, int64_t n_rows, int d, int k,
                                   int m_keep, int fill, float scale2,
                                   void *stream_) {
    if (n < 0 || n_rows < 1 || k < 1 || k > 256 || m_keep < 1) return PA_E_SHAPE;
    if (d <= 0 || d % kChunk) return PA_E_DIM;
    if (n == 0) return PA_OK;
    if (!selected || !rows_hi_f16 || !rows_lo_f16 || !norm || !cand || !cand_dist)
        return PA_E_NULL;
    PruneRowsArgs a;
    a.hi = reinterpret_cast<const _Float16 *>(rows_hi_f16);
    a.lo = reinterpret_cast<const _Float16 *>(rows_lo_f16);
    a.norm = norm, a.cand = cand, a.cand_dist = cand_dist, a.selected = selected;
    a.n = n, a.n_rows = n_rows, a.d = d, a.k = k, a.m_keep = m_keep, a.fill = fill;
    a.scale2 = scale2;
    // a launch holds fewer than 2^32 work-items: at most 2^22 nodes of 256
    for (a.first = 0; a.first < n; a.first += kLaunchNodes) {
        const int64_t count = n - a.first < kLaunchNodes ? n - a.first : kLaunchNodes;
        prune_rows_kernel<<<(unsigned)count, 256, 0, (hipStream_t)stream_>>>(a);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return (int)err;
    }
    return PA_OK;
}

extern "C" int pa_graph_prune(int32_t *selected, const float *pair,
                              const float *cand_dist, int64_t n, int k,
                              int m_keep, int fill, void *stream_) {
    if (n < 0 || k < 1 || k > 512 || m_keep < 1) return PA_E_SHAPE;
    if (n >= (1ll << 32) / kWave) return PA_E_RANGE;   // work-items of the launch
    if (n == 0) return PA_OK;
    if (!selected || !pair || !cand_dist) return PA_E_NULL;
    prune_kernel<<<(unsigned)((n + 3) / 4), 256, 0, (hipStream_t)stream_>>>(
        pair, cand_dist, selected, n, k, m_keep, fill);
    return (int)hipGetLastError();
}
