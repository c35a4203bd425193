// Rings inside a compute unit: the ring collectives of ring.hpp with all
// positions of a ring in one lane and the hops between them in its registers.
//
// The walks of ring.hpp put neighbouring positions on different compute units
// and their staging into the L2 of an XCD.  A hop then costs a 1 KiB store and
// a 1 KiB load through the L2 beside the rows from HBM, and a compute unit
// keeps only some 130 requests in flight: an 8-rank reduce-scatter spends half
// of its time on staging.  Virtual ranks share one GPU, so one lane can stand
// at every position in turn: it loads its 16 bytes of every rank's row, all of
// them at once, walks the ring from the pipeline's root with the partial sum in
// registers - the additions and their order are those of the hops - and stores
// the result at the positions that keep it.  Each row crosses the memory system
// once; there is no staging, no epoch, no seat to claim and nobody to wait for,
// and both protocols (which say how a hop is made safe) are the same.
//
// Bound by HBM (6.4 - 7.0 TB/s of rows read and written).  A thread block moves
// one tile and ends, and the tiles of a pipeline follow each other in the order
// the blocks are dealt: what is in flight over the device is one window of
// consecutive bytes per row that moves through memory.  Wavefronts that stay
// resident and stride through the rows drift apart and lose a tenth of the rate.
// 8 ranks: one ring per resident thread block, hops through LDS / one lane and
// resident / a block per tile / and the wavefronts held down (cu_waves):
// reduce-scatter of 256 MiB f16 447 / 470 / 391 / 375 us, allgather of 8 x 128 MiB
// 1675 / 1660 / 1540 / 1380 (4 KiB to a wavefront 1318), allreduce of 64 MiB bf16 205 / 198 /
// 190 / 161.
#pragma once
#include <type_traits>
#include <utility>

#include "ring.hpp"

namespace mint {

// One launch.  Grid: tiles of a row, then one block for its ragged ends if it has
// any, and pipelines (alltoall: destinations) in x and y (CuPlace); the sources of an
// alltoall in z.
//
// A block lives for one trip to memory, so what it does before its loads are out
// counts: the numbers come as the first kernel arguments, which the compiler has the
// hardware put into scalar registers before the first instruction (kernarg preload;
// not what is inside a struct, hence the vector), and one round of scalar loads brings
// the addresses.  Few of them, since each argument costs a launch 10 ns.
struct CuShape {
    uint64_t row_bytes, row_stride;
    uint64_t short_bytes;          // bytes of row `full`; rows behind it are empty
    uint32_t starts;               // bits 3 p: index in the ring of pipeline p's root
    uint32_t full;                 // rows before this one have row_bytes
    uint32_t tiles;                // thread blocks that share the whole vectors of a row
    uint32_t part;                 // small form: tiles of a row that one XCD takes, or 0 (CuPlace);
                                   // large form: cu_pause of a wavefront before it stores

    CuShape() = default;
    __device__ __forceinline__ CuShape(u64x4 numbers, u32x2 counts)
        : row_bytes(numbers.x), row_stride(numbers.y), short_bytes(numbers.z), starts((uint32_t)numbers.w),
          full((uint32_t)(numbers.w >> 32)), tiles(counts.x), part(counts.y) {}
    void numbers(u64x4& x) const { x = u64x4{row_bytes, row_stride, short_bytes, (uint64_t)full << 32 | starts}; }
};

// The ranks' buffers in the order of the ring.  One address per rank where they
// work in place, as the operators do: a launch with up to 112 bytes of arguments
// takes the host 2.7 us, one with more 3.3 - 3.5.  SPLIT: N addresses to load from, then
// N to store to.
template <int N, bool SPLIT>
struct CuTables {
    uint64_t rank[SPLIT ? 2 * N : N];
    uint64_t* status;
};
static_assert(sizeof(CuShape) + sizeof(CuTables<kMaxRanks, false>) <= 112, "arguments of a launch in place");

// The ranks' buffers where ranks work in place and all rows lie within 4 GiB (`near` in
// CuRingArgs): the lowest address and every rank's distance from it, in bytes.  With numbers
// of 32 bits all that the loads wait for fits into the 14 words that a launch can bring in
// registers (of seven and eight ranks the status block's address comes behind them and is read from memory, by the one
// wavefront that looks there).  A table in memory costs each block a round trip before its
// loads, and its compute unit's first blocks a long one: the runtime has just written it across the bus.
// Over launches by tables, us, trains of calls over three sets of buffers in turn:
//   touched      10 MiB        25 MiB        64 MiB        110 MiB        400 MiB
//   8 ranks, allgather       2.95 / 2.67   4.65 / 4.23   9.38 / 8.85   17.0 / 16.8    57.9 / 57.3
//            reduce-scatter  2.74 / 2.53   5.49 / 5.25   11.2 / 10.9   23.7 / 22.7    68.7 / 68.2
//            allreduce       4.19 / 3.93   8.49 / 8.06   18.8 / 18.8   40.6 / 40.6    130 / 129
//   3 ranks, broadcast       2.57 / 2.51   3.79 / 3.60   10.2 / 10.1   16.9 / 16.8    63.2 / 62.1
//            reduce          3.44 / 3.45   6.13 / 6.07   13.2 / 13.1   22.3 / 22.1    85.6 / 83.6
// Below 4 MiB the host's 2.7 us per launch hide it.
//   rows    lowest address (two words), row_bytes, row_stride; where rows are cut (kCuNearCut),
//           which follow each other without gaps then, short_bytes in its place; distances of
//           ranks 0 - 3
//   high    those of the ranks from 4 on
//   counts  starts | full << 24 | kCuNearCut, tiles | part << 16 (large form: << 24)
//   status
// Each argument costs a launch 10 ns, so what follows the rows shares one where it fits
// (cu_near_more): up to four ranks {counts, status}; five and six {high, counts}, status; seven
// and eight high, counts, status.
constexpr uint32_t kCuNearCut = 1u << 31;
// At most: bytes from the lowest address to the end of the last row, of a row (offsets have a
// sign), tiles of a row in the small form.
constexpr uint64_t kCuNearSpan = 0xffffffffull, kCuNearRow = 1ull << 30;
constexpr uint32_t kCuNearTiles = 0xffff;
constexpr uint32_t cu_near_part_bit(bool large) { return large ? 24u : 16u; }
static_assert(kCuNearRow / 1024 + 1 < 1u << cu_near_part_bit(true), "tiles of a KiB in the large form");

// (host side: the whole of a launch)
struct CuRingArgs {
    CuShape shape;
    uint64_t input[kMaxRanks], output[kMaxRanks];
    uint64_t* status;
    uint32_t op, pipes, len;
    uint32_t blocks;               // of the grid for the tiles of a row and its ends
    bool split;
    uint64_t lowest;               // of the ranks' addresses
    bool near;
};

// How rows are loaded: through the caches, or streamed past the last-level one.
template <bool STREAM>
__device__ __forceinline__ u32x4 cu_load(const uint8_t* uniform, uint32_t lane) {
    MINT_GLOBAL const u32x4_unaligned* const p = (MINT_GLOBAL const u32x4_unaligned*)(as_global(uniform) + lane);
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    else return *p;
}
// How results are stored: past the last-level cache (nt), through the XCD's L2
// (sc1), or both.  8 ranks, kept in the L2 / nt / sc1 / sc1 nt:
//   small, a row to several places: allgather of 8 x 8 MiB  9.9 / 10.5 /  8.2 / 10.1 us
//   small, a row to one place:      sendrecv of 48 MiB     18.8 / 13.7 / 16.4 / 13.4
//   large, several:                 allgather of 8 x 64 MiB   - / 73.4 / 94.3 / 67.7
//   large, one:                     reduce-scatter of 64 MiB 86.9 / 88.6 / 82.1 / 88.0
enum { CU_NT = 0, CU_SC1 = 1, CU_SC1_NT = 2 };
// A copy to one place in the small form, up to 24 MiB touched: sc1.  The results stay
// in the L2s, and the kernel that reads them next takes 6 - 20 us less than behind nt or sc1 nt
// (multiplied in place, buffers of 3 - 6 MiB 27 -> 7 us and 13 -> 7); alone the call takes 0.94 / 0.96 / 1.03 -
// 1.07 of nt (the same buffers again / three sets in turn / buffers that 700 MiB lie between two uses of).
// (a pipeline to each XCD leaves a whole row of results in one XCD's L2: short ones, which few blocks
// read next, are sooner there from the last-level cache.  Alltoall of eight ranks, multiplied in place
// behind the call, sc1 / nt: 2 MiB 4 us more, 2.5 MiB 6 less)
// Beyond: sc1 nt, a choice that holds whatever the caches hold, nt alone does not (with eight pipelines,
// a pipeline to each XCD, it does: odd rows 1.00 / 1.06 / 1.06 by sc1 nt).  Alltoall of 2 to 7 ranks, over
// nt in tiles dealt one by one, tiles dealt by the eighth (CuPlace):
//   touched MiB       25 - 30               30 - 64               65 - 160
//   nt         0.83 / 0.94 / 1.03    0.81 / 0.94 / 1.02    0.96 / 0.95 / 0.99
//   sc1 nt     0.86 / 0.94 / 1.00    0.80 / 0.94 / 0.98    0.93 / 0.94 / 0.96
// sendrecv and the copies of two ranks alike (65 - 160 MiB nt 0.97 / 0.98 / 1.02, sc1 nt 0.97 / 0.97 / 1.00).
//
// A sum to one place in the small form: sc1 in the bands below (cu_through_mib), nt elsewhere.  Time over
// that of nt in tiles dealt one by one, reduce and reduce-scatter in three types, the same buffers again /
// three sets in turn / 700 MiB between two uses, geometric means (largest):
//   touched MiB              sc1                                        nt
//   2 ranks   4 - 6   0.98 (1.05) / 1.01 (1.09) / 1.02 (1.06)    0.96 (1.01) / 0.98 (1.02) / 0.99 (0.99)
//             6 - 20  0.89 (1.02) / 0.87 (1.02) / 1.00 (1.05)    0.96 (1.00) / 0.99 (1.09) / 1.00 (1.07)
//            32 - 56  0.73 (0.89) / 0.94 (0.97) / 0.99 (1.05)    1.00 (1.13) / 0.98 (1.02) / 1.02 (1.09)
//   3 ranks   6 - 12  0.98 (1.03) / 0.93 (1.03) / 1.08 (1.51)    0.97 (1.00) / 0.98 (1.02) / 0.99 (1.00)
//            12 - 20  0.91 (0.98) / 0.87 (1.01) / 0.99 (1.02)    0.98 (1.00) / 0.99 (0.99) / 0.99 (1.00)
//            32 - 56  0.77 (1.01) / 0.93 (0.99) / 0.97 (1.03)    0.97 (1.08) / 0.94 (1.00) / 0.99 (1.05)
//   4 - 8     4 - 20  0.98 (1.11) / 0.97 (1.05) / 1.00 (1.32)    0.97 (1.02) / 0.98 (1.03) / 0.99 (1.02)
//   4 - 7    20 - 32  0.90 (1.11) / 0.96 (1.03) / 0.98 (1.05)    0.88 (1.07) / 0.95 (1.01) / 0.98 (1.05)
//            32 - 56  0.87 (1.13) / 0.96 (1.04) / 0.97 (1.05)    0.97 (1.31) / 0.95 (1.03) / 0.98 (1.09)
// sc1 takes longest on rows of 2 - 3 MiB that lie 4 MiB apart and are in no cache: 3 ranks 3.6 -> 5.9
// us, 4 ranks 4.3 -> 5.8.  With a pipeline to each XCD it is 1.08 / 1.01 / 1.00 at 20 - 32 MiB.
//
// Not taken for either: rows streamed.  The call alone is then 0.85 - 0.95 of that at 12 - 40 MiB, but
// streamed rows do not stay in any cache.  A kernel that reads the buffers again next takes 8 - 13 us
// longer (multiplied in place, four ranks of 22 MiB in all 17 -> 25 us), and the same call on the same
// buffers again up to 1.3 at 20 - 32 MiB.
struct CuBand {
    int above, most;          // MiB touched
};
constexpr CuBand cu_through_mib(bool sums, int ranks, int pipes, bool pipe_each) {
    if (!sums) return {pipe_each ? 2 : 0, 24};
    if (ranks <= 3) return {ranks == 2 ? 6 : 12, 1 << 20};
    if (pipe_each || (ranks >= 7 && pipes == 1)) return {0, 0};      // (cu_by_eighths)
    return {32, 56};
}
// Sums to one place that are far larger than the last-level cache (plan_cu): with
// many rows to read nt is the faster one, on buffers that have not just been used.
// Four sets of buffers in turn, reduce-scatter and reduce of f16 and bf16, nt over
// sc1: 0.94 - 1.01 for 6, 7 and 8 ranks at 560 MiB touched and up; three sets, f16
// reduce-scatter, sc1 / nt, us, 8 / 7 / 6 / 5 / 4 ranks (f32 the same):
//   448 MiB  75 / 80,  77 / 82,  80 / 86,  84 / 88,  90 / 96;
//   800     144 / 141, 152 / 145, 154 / 151, 153 / 156, 158 / 168;
//   1 GiB   181 / 179, 192 / 185, 198 / 194, 200 / 200, 204 / 213;
//   2 GiB   386 / 378, 381 / 369, 401 / 391, 410 / 399, 415 / 428.
// The same buffers again and again keep a part of the sums in the cache with sc1:
// there nt takes 1 - 11 % longer up to 1.5 GiB and is ahead from 2.3 GiB on.
constexpr int kCuStreamRanks = 6;
// Sums to one place of two to six ranks, rows up to cu_mid_mib touched: the places of
// the small form, rows streamed past the last-level cache, results left in it (the rows
// of three sets of buffers are beyond it, their results are not).  5 and 6 ranks in blocks of 64 threads, 14
// wavefronts on a compute unit; 4 ranks: cu_mid_waves.  Over the large form with its waits (cu_pauses), reduce and
// reduce-scatter in three types, geometric means, the same buffers again / three sets in turn / 700 MiB between two uses /
// 3.5 GB between two uses:
//   touched MiB     100 - 120                  120 - 145                  145 - 165                  165 - 190                  190 - 264
//   2 ranks  0.96 / 0.96 / 1.04 / 1.04  0.97 / 0.98 / 1.03 / 1.03  0.99 / 0.98 / 1.04 / 1.04  0.99 / 0.98 / 1.04 / 1.05  1.01 / 1.03 / 1.03 / 1.04
//   3        0.93 / 0.96 / 1.00 / 1.03  0.94 / 0.97 / 1.06 / 1.07  0.98 / 0.97 / 1.04 / 1.05  1.01 / 0.98 / 1.06 / 1.07  1.00 / 0.99 / 1.07 / 1.08
//   4        0.92 / 0.98 / 0.98 / 1.02  0.93 / 1.01 / 1.01 / 1.03  1.01 / 1.00 / 1.01 / 1.05  1.02 / 0.99 / 1.00 / 1.05  1.04 / 0.99 / 1.00 / 1.05
//   5        0.96 / 0.98 / 0.98 / 1.01  0.98 / 1.02 / 1.00 / 1.05  0.99 / 1.02 / 1.00 / 1.04  1.06 / 1.02 / 1.00 / 1.04
//   6        0.95 / 1.00 / 0.99 / 1.02  0.97 / 1.01 / 1.00 / 1.03  1.02 / 1.02 / 1.01 / 1.05
// The lines stand where the form crossed the large one without waits (at 176 MiB 0.97 throughout): with them it is ahead up to
// about 140 MiB, and on distant uses nowhere.
constexpr int kCuMidRanks = 6;
constexpr int cu_mid_mib(int ranks) {
    return ranks == 2 ? 196 : ranks == 3 ? 264 : ranks == 4 ? 208 : ranks == 5 ? 176 : 160;
}

// Rows of six and more ranks to several places (VAST below) from so many MiB touched
// on.  Over the large form at 0.9 / 1.5 / 3 / 4 GiB touched, three sets of buffers in turn:
// allgather of 6 ranks 1.01 / 0.98 / 0.95 / 0.94, 7 ranks 0.96 / 0.96 / 0.94 / 0.94, 8 ranks
// 1.00 / 0.99 / 0.97 / 0.95 (6 and 8 GiB 0.95 / 0.94); 5 ranks 1 - 2 % slower throughout.
constexpr int kCuVastCopies = 6;
constexpr int cu_vast_mib(int ranks) { return ranks == 7 ? 700 : ranks == 6 ? 1280 : 2560; }

// The forms of a launch (which: plan_cu in mintccl.hip).
//
// LARGE, rows beyond the last-level cache: one wavefront per block and 1 KiB
// tiles that begin at whole KiB, the pipelines one after the other, as few
// wavefronts on a compute unit as keep HBM busy (cu_waves).  More of them widen
// the window over which the loads and stores of 8 or 16 rows are scattered: 8
// ranks, reduce-scatter of 256 MiB 392 us with 32 to a compute unit, 376 with 9;
// allreduce of 64 MiB 202 with 20, 158 with 4; allgather of 8 x 64 MiB 89 with 32,
// 67 with 8.  Rows to several places, over blocks of 128 threads and 2 KiB, three sets
// of buffers in turn: allgather of 3 / 4 / 5 / 6 / 7 ranks at 0.1 - 2 GiB touched 0.98 /
// 0.99 / 0.98 / 0.97 / 0.96; eight ranks lose 1 - 5 % by it and keep those.  Tiles at
// whole KiB rather than lines: ragged rows 1 %.
//
// VAST, rows of six and more ranks to several places, far beyond the cache
// (kCuVastCopies): a wavefront moves 4 KiB, all of it loaded at once and every KiB
// stored at all places before the next, four or five wavefronts on a compute unit.
// HBM takes seven streams of rows the better the longer the stretches are that
// arrive: 8 ranks, allgather of 8 x 128 MiB 1405 -> 1318 us (1473 -> 1331 with rows that
// are no multiple of a line), 7 ranks and 4 GiB 0.94, 6 ranks 0.96.
//
// SMALL, otherwise: blocks of 128 threads and 2 KiB, loads through the cache, to each XCD
// consecutive tiles (CuPlace).  8 ranks, reduce-scatter of 8 MiB 10.9 us, 15.5 in the
// large form.  Blocks of 64 and of 256 threads with 2 KiB and 4 KiB are within 1 % of
// it, 4 KiB by 64 threads 2 - 4 % slower, 512 threads up to a tenth where rows are added.
// CuMidSum (kCuMidRanks) is the small form in its places, with the large one's loads.
template <int THREADS, int VECTORS, bool LARGE, bool STREAM, int STORES>
struct CuForm {
    static constexpr int kThreads = THREADS;       // of a block
    static constexpr int kVectors = VECTORS;       // of 16 bytes a thread moves, THREADS of them apart
    static constexpr uint32_t kTile = THREADS * VECTORS * 16;
    static constexpr bool kLarge = LARGE;
    static constexpr uint32_t kAlign = LARGE ? 1023 : 127;   // a tile begins at a multiple of kAlign + 1
    static constexpr bool kStream = STREAM;        // rows are loaded past the last-level cache
    static constexpr int kStores = STORES;
};
template <int STORES>
using CuSmall = CuForm<128, 1, false, false, STORES>;
template <int N>
using CuMidSum = CuForm<N <= 4 ? 128 : 64, 1, false, true, CU_SC1>;   // (kCuMidRanks)
using CuLargeSum = CuForm<64, 1, true, true, CU_SC1>;            // to one place
using CuLargeSumStreamed = CuForm<64, 1, true, true, CU_NT>;     // (kCuStreamRanks)
using CuLargeSumEverywhere = CuForm<64, 1, true, true, CU_SC1_NT>;
using CuLargeCopy = CuForm<64, 1, true, true, CU_SC1>;           // to one place
template <int N>
using CuLargeCopies = CuForm<N == 8 ? 128 : 64, 1, true, false, CU_SC1_NT>;    // to several
using CuVastCopies = CuForm<64, 4, true, false, CU_SC1_NT>;

// What plan_cu decides by the sizes of a launch, and the form that this makes of it: the
// one place where a form is named, for the grid that plan_cu counts and for the kernel that
// is launched alike.
struct CuChoice {
    bool large, far;          // rows beyond the last-level cache, far beyond it
    bool mid;                 // neither: CuMidSum
    bool through;             // small: cu_through_mib
    bool pipe_each;           // small: each XCD takes a pipeline (CuPlace)
};
// (IN_PLACE: ranks that work in place are given by one address each; to a launch beyond the
// small form the host's time is nothing)
template <typename FORM, bool IN_PLACE = !FORM::kLarge>
struct CuFormIs {
    using type = FORM;
    static constexpr bool in_place = IN_PLACE;
};
// use(CuFormIs<form>{}), sums of N ranks
template <int N, bool EVERYWHERE, typename USE>
auto cu_sum_form(const CuChoice& c, const USE& use) {
    if constexpr (EVERYWHERE) {
        return c.large ? use(CuFormIs<CuLargeSumEverywhere>{}) : use(CuFormIs<CuSmall<CU_SC1>>{});
    } else {
        if constexpr (N >= kCuStreamRanks)
            if (c.far) return use(CuFormIs<CuLargeSumStreamed>{});
        if constexpr (N <= kCuMidRanks)
            if (c.mid) return use(CuFormIs<CuMidSum<N>, false>{});
        if (c.large) return use(CuFormIs<CuLargeSum>{});
        return c.through ? use(CuFormIs<CuSmall<CU_SC1>>{}) : use(CuFormIs<CuSmall<CU_NT>>{});
    }
}
// a row copied to one place (sendrecv, alltoall, two ranks)
template <typename USE>
auto cu_move_form(const CuChoice& c, const USE& use) {
    if (c.large) return use(CuFormIs<CuLargeCopy>{});
    if (c.through) return use(CuFormIs<CuSmall<CU_SC1>>{});
    return c.pipe_each ? use(CuFormIs<CuSmall<CU_NT>>{}) : use(CuFormIs<CuSmall<CU_SC1_NT>>{});
}
// a row of N ranks copied to the others
template <int N, typename USE>
auto cu_copy_form(const CuChoice& c, const USE& use) {
    if constexpr (N == 2) {
        return cu_move_form(c, use);
    } else {
        if constexpr (N >= kCuVastCopies)
            if (c.far) return use(CuFormIs<CuVastCopies>{});
        return c.large ? use(CuFormIs<CuLargeCopies<N>>{}) : use(CuFormIs<CuSmall<CU_SC1>>{});
    }
}
// use(CuCount<ranks>{}), or MINT_ERR_ARG
template <int N>
struct CuCount {
    static constexpr int value = N;
};
template <typename USE>
int cu_with_ranks(int ranks, const USE& use) {
    switch (ranks) {
        case 2: return use(CuCount<2>{});
        case 3: return use(CuCount<3>{});
        case 4: return use(CuCount<4>{});
        case 5: return use(CuCount<5>{});
        case 6: return use(CuCount<6>{});
        case 7: return use(CuCount<7>{});
        case 8: return use(CuCount<8>{});
        default: return MINT_ERR_ARG;
    }
}

template <int HOW>
__device__ __forceinline__ void cu_store(uint8_t* uniform, uint32_t lane, u32x4 v) {
    if constexpr (HOW == CU_NT)
        __builtin_nontemporal_store(v, (MINT_GLOBAL u32x4_unaligned*)(as_global(uniform) + lane));
    else
        st128_through<HOW == CU_SC1_NT>(uniform, lane, v);
}

// A row cut into vectors of 16 bytes whose stores are aligned: vector i covers
// the bytes from 16 i - `shift` on.  Vectors that are not wholly inside the row
// are left out; the bytes they would have brought, fewer than 16 at either end,
// are moved one element per lane.
// WIDE: offsets in a row may need more than 31 bits, and tiles more blocks than a grid has.
template <typename FORM, bool WIDE = FORM::kLarge>
struct CuRow {
    using Bytes = std::conditional_t<WIDE, uint64_t, uint32_t>;
    using Offset = std::conditional_t<WIDE, int64_t, int32_t>;
    Bytes bytes;
    uint32_t shift;
    __device__ __forceinline__ CuRow(uint64_t row_bytes, uint64_t short_bytes, uint32_t full, uint32_t p,
                                     const uint8_t* stored, uint32_t size) {
        bytes = p < full ? (Bytes)row_bytes : p == full ? (Bytes)short_bytes : 0u;
        // (whole elements: a row may start at any byte)
        shift = (uint32_t)(uintptr_t)stored & FORM::kAlign & ~(size - 1u);
    }
    // Element of `size` bytes that this lane (of the first 32) moves, or none.
    __device__ __forceinline__ bool end_element(uint32_t size, Bytes& off) const {
        uint32_t head = (0u - shift) & 15u;
        head = bytes < head ? (uint32_t)bytes : head;
        const uint32_t tail = (uint32_t)(bytes - head) & 15u;
        const uint32_t at = (threadIdx.x & 15u) * size;
        const bool first = threadIdx.x < 16u;
        off = first ? at : bytes - tail + at;
        return threadIdx.x < 32u && at < (first ? head : tail);
    }
    // The vectors of a tile: walk(offset of the block's first, how many of them a
    // lane has), all at once where all are wholly inside the row.
    template <typename WALK>
    __device__ __forceinline__ void tile(uint64_t t, const WALK& walk) const {
        const Offset base = (Offset)((Bytes)t * FORM::kTile) - (Offset)shift;
        if constexpr (FORM::kVectors > 1)
            if (base >= 0 && (Bytes)base + FORM::kTile <= bytes) {
                walk(base, CuCount<FORM::kVectors>{});
                return;
            }
        // (lane by lane: a compute unit has one scalar unit for all its wavefronts)
#pragma unroll 1
        for (int i = 0; i < FORM::kVectors; ++i) {
            const Offset off = base + i * FORM::kThreads * 16, mine = off + (Offset)(threadIdx.x * 16u);
            if (mine >= 0 && (Bytes)mine + 16u <= bytes) walk(off, CuCount<1>{});
        }
    }
    template <typename WALK>
    __device__ __forceinline__ void tiles(uint32_t mine, uint32_t all, const WALK& walk) const {
        if constexpr (WIDE)
            for (uint64_t t = mine; t * FORM::kTile < bytes + shift; t += all) tile(t, walk);
        else
            tile(mine, walk);
    }
};

// (device side of a launch by distances)
struct CuNear {
    uint8_t* lowest;
    uint32_t row_bytes, row_stride, short_bytes;
    u32x8 rank;
    uint32_t starts, full, tiles, part;
    uint64_t* status;
    __device__ __forceinline__ CuNear(bool large, u32x8 rows, u32x4 high, u32x2 counts, uint64_t* status_)
        : lowest(reinterpret_cast<uint8_t*>((uint64_t)rows[1] << 32 | rows[0])), row_bytes(rows[2]),
          row_stride(counts.x & kCuNearCut ? rows[2] : rows[3]), short_bytes(rows[3]),
          rank{rows[4], rows[5], rows[6], rows[7], high.x, high.y, high.z, high.w}, starts(counts.x),
          full(counts.x >> 24 & 15u), tiles(counts.y & ((1u << cu_near_part_bit(large)) - 1u)), part(counts.y >> cu_near_part_bit(large)),
          status(status_) {}
    __device__ __forceinline__ CuNear(bool large, u32x8 rows, u32x4 words, uint64_t* status_)
        : CuNear(large, rows, u32x4{words.x, words.y, 0u, 0u}, u32x2{words.z, words.w}, status_) {}
    __device__ __forceinline__ CuNear(bool large, u32x8 rows, u32x4 words)
        : CuNear(large, rows, u32x4{}, u32x2{words.x, words.y}, reinterpret_cast<uint64_t*>((uint64_t)words.w << 32 | words.z)) {}
    __device__ __forceinline__ uint32_t root(uint32_t p) const { return starts >> (3u * p) & 7u; }
    template <typename FORM>
    __device__ __forceinline__ CuRow<FORM, false> row(uint32_t p, const uint8_t* stored, uint32_t size) const {
        return CuRow<FORM, false>(row_bytes, short_bytes, full, p, stored, size);
    }
};

// Where a block works.  The hardware deals consecutive blocks to the eight XCDs in
// turn.  Large form: one row after the other, all XCDs next to each other.  Small
// form: consecutive tiles are one XCD's affair - an eighth of every row (`part` tiles;
// a row begins on another XCD than the one before it) or, where the pipelines are a
// multiple of eight, a pipeline.  Against tiles dealt one by one, ranks 2 to 7,
// geometric means over 24 - 48 MiB / 64 - 96 MiB touched, three sets of buffers in turn:
// sendrecv 0.90 / 0.94, alltoall 0.94 / 0.96, reduce 0.95 / 0.97, reduce-scatter 0.95 /
// 0.96, broadcast 0.94 / 0.99, allgather 0.96 / 0.98, allreduce 0.93 / 0.96.  Eight
// pipelines: an eighth of every row 1.03 (alltoall), 1.00 (reduce-scatter) and 1.02
// (allgather) of a pipeline to each.
//
// The tile of block x of a row whose first tiles are XCD `turn`'s (mod 8), `part` tiles to each XCD:
__host__ __device__ constexpr uint32_t dealt_tile(uint32_t x, uint32_t turn, uint32_t part) {
    return ((x + turn) & 7u) * part + (x >> 3);
}
// (8 part blocks have as many tiles, each once)
constexpr bool dealt_once(uint32_t part) {
    for (uint32_t turn = 0; turn < 2 * 8; ++turn) {
        bool taken[64] = {};
        for (uint32_t x = 0; x < 8 * part; ++x) {
            const uint32_t tile = dealt_tile(x, turn, part);
            if (tile >= 8 * part || taken[tile]) return false;
            taken[tile] = true;
        }
    }
    return true;
}
static_assert(dealt_once(1) && dealt_once(2) && dealt_once(3) && dealt_once(5) && dealt_once(8), "one block per tile");
struct CuPlace {
    uint32_t tile, pipe;
    __device__ __forceinline__ CuPlace(bool large, uint32_t part) {
        const uint32_t x = blockIdx.x, y = blockIdx.y;
        if (large) {
            tile = x;
            pipe = y;
        } else if (part) {
            tile = dealt_tile(x, y + blockIdx.z, part);
            pipe = y;
        } else {
            tile = y;
            pipe = x;
        }
    }
};

// A launch that finds the abort flag of its status block set (an earlier launch
// through staging gave up) is counted there, as in take_seat; by the last
// wavefront of the first block, which has nothing else to do in a launch so
// small that this load would show.
template <uint32_t THREADS>
__device__ __forceinline__ void cu_count_if_aborted(uint64_t* status) {
    if (__builtin_expect((blockIdx.x | blockIdx.y | blockIdx.z) == 0u, 0) && threadIdx.x >= THREADS - 64u)
        count_launch_if_aborted(status, 0);
}

typedef uint32_t u32_unaligned __attribute__((aligned(1)));
typedef uint16_t u16_unaligned __attribute__((aligned(1)));
template <int DT>
__device__ __forceinline__ uint32_t cu_load_element(const uint8_t* p) {
    if constexpr (DT == DT_BYTES) return *as_global(p);
    else if constexpr (DT == DT_F32) return *(MINT_GLOBAL const u32_unaligned*)p;
    else return *(MINT_GLOBAL const u16_unaligned*)p;
}
template <int DT>
__device__ __forceinline__ void cu_store_element(uint8_t* p, uint32_t v) {
    if constexpr (DT == DT_BYTES) *as_global(p) = (uint8_t)v;
    else if constexpr (DT == DT_F32) *(MINT_GLOBAL u32_unaligned*)p = v;
    else *(MINT_GLOBAL u16_unaligned*)p = (uint16_t)v;
}

// Where the addresses have to be there: the compiler would fetch each where it is
// first used, a scalar load and a wait at a time.
template <int N, typename P>
__device__ __forceinline__ void cu_here(P* (&x)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+s"(x[i]));
}
// The addresses of a table from `root` on around the ring (by their bytes' distance from
// its start, which one scalar load takes as it is).
template <int N>
__device__ __forceinline__ void cu_around(const uint64_t* table, uint32_t root, const uint8_t* (&x)[N]) {
    uint32_t at = root * 8u;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        x[i] = *reinterpret_cast<const uint8_t* const*>(reinterpret_cast<const uint8_t*>(table) + at);
        at = at == 8u * (N - 1) ? 0u : at + 8u;
    }
    cu_here(x);
}

// Where a block finds the ranks' rows: ranks as they follow each other around the ring, the
// pipeline's root first; an offset in a row is a part that all lanes share and a lane's.
//
// By their addresses.  STORED: places that are stored to, the root's first.
template <int N, int STORED>
struct CuByTable {
    const uint8_t* from[N];
    uint8_t* to[STORED];
    uint64_t row_off;
    // (a uniform part and a lane's: scalar base and 32-bit offset of one instruction)
    template <bool STREAM>
    __device__ __forceinline__ u32x4 load(int h, int64_t off, uint32_t lane) const {
        return cu_load<STREAM>(from[h] + ((int64_t)row_off + off), lane);
    }
    template <int HOW>
    __device__ __forceinline__ void store(int i, int64_t off, uint32_t lane, u32x4 v) const {
        cu_store<HOW>(to[i] + ((int64_t)row_off + off), lane, v);
    }
    template <int DT>
    __device__ __forceinline__ uint32_t load_element(int h, uint64_t off) const { return cu_load_element<DT>(from[h] + row_off + off); }
    template <int DT>
    __device__ __forceinline__ void store_element(int i, uint64_t off, uint32_t v) const { cu_store_element<DT>(to[i] + row_off + off, v); }
};
// By their distances from the lowest of them (CuNear).
// FIRST: the first rank that is stored to.
template <int N, int FIRST>
struct CuByDistance {
    // (a vector, not an array: of that the compiler would make LDS for an index it finds in
    // the selects)
    typedef uint32_t Ranks __attribute__((ext_vector_type(N)));
    uint8_t* lowest;
    Ranks rank;
    uint32_t row_off;
    template <int BY, int... I>
    static __device__ __forceinline__ Ranks turned(Ranks x, std::integer_sequence<int, I...>) {
        return __builtin_shufflevector(x, x, (I + BY) % N...);
    }
    // turned by the bits of `root`: one select of two scalars per rank and bit
    template <int BY = 1>
    static __device__ __forceinline__ Ranks around(Ranks x, uint32_t root) {
        if constexpr (BY >= N) return x;
        else return around<2 * BY>(root & BY ? turned<BY>(x, std::make_integer_sequence<int, N>{}) : x, root);
    }
    __device__ __forceinline__ CuByDistance(const CuNear& a, uint32_t root, uint32_t row_off_) : lowest(a.lowest), row_off(row_off_) {
        Ranks x;
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = a.rank[i];
        if (root) {
            // (a branch: the one row of a reduce or a broadcast is named from its root on.  8 ranks, reduce and
            // broadcast of 6 - 25 MiB touched 0.98 - 0.99, beyond and allgather 1.00)
            asm volatile("");
            x = around(x, root);
        }
        rank = x;
    }
    __device__ __forceinline__ const uint8_t* stored() const { return lowest + rank[FIRST] + row_off; }
    template <bool STREAM>
    __device__ __forceinline__ u32x4 load(int h, int32_t off, uint32_t lane) const {
        return cu_load<STREAM>(lowest, rank[h] + (row_off + (uint32_t)off + lane));
    }
    template <int HOW>
    __device__ __forceinline__ void store(int i, int32_t off, uint32_t lane, u32x4 v) const {
        cu_store<HOW>(lowest, rank[FIRST + i] + (row_off + (uint32_t)off + lane), v);
    }
    template <int DT>
    __device__ __forceinline__ uint32_t load_element(int h, uint32_t off) const {
        return cu_load_element<DT>(lowest + (rank[h] + (row_off + off)));
    }
    template <int DT>
    __device__ __forceinline__ void store_element(int i, uint32_t off, uint32_t v) const {
        cu_store_element<DT>(lowest + (rank[FIRST + i] + (row_off + off)), v);
    }
};

// A wavefront of the large form that has its rows waits `times` 256 clocks before it stores
// (cu_pauses in mintccl.hip: how often, and what it is worth).
__device__ __forceinline__ void cu_pause(uint32_t times, u32x4& arrived) {
#pragma unroll 1
    for (; times; --times) asm volatile("s_sleep 4" : "+v"(arrived));
}

// Rings that add: N ranks, the sum goes to the root of the pipeline (reduce,
// reduce-scatter) or to all of them (allreduce): to STORED places.
template <int DT, int N, int STORED, typename FORM, bool WIDE, typename PLACES>
__device__ __forceinline__ void cu_sum_row(const CuRow<FORM, WIDE>& row, uint32_t tile, uint32_t tiles, uint32_t pauses, const PLACES& at) {
    using Row = CuRow<FORM, WIDE>;
    if (__builtin_expect(tile < tiles, 1)) {
        const uint32_t lane = threadIdx.x * 16u;
        row.tiles(tile, tiles, [&](typename Row::Offset base, auto count) MINT_INLINE_LAMBDA {
            constexpr int kCount = decltype(count)::value, kStep = FORM::kThreads * 16;
            u32x4 v[kCount][N];
#pragma unroll
            for (int k = 0; k < kCount; ++k)
#pragma unroll
                for (int h = 0; h < N; ++h) v[k][h] = at.template load<FORM::kStream>(h, base + k * kStep, lane);
#pragma unroll
            for (int k = 0; k < kCount; ++k) {
                // (three ranks of bf16 in the large form: the longer additions are a part of the wait before the stores
                // (cu_pauses), 0.990 - 0.995 of the shorter ones at 270 - 700 MiB touched, 0.998 at 1000, and no wait of
                // whole 256 clocks in their place does it)
                Sum<DT, FORM::kLarge && N == 3 && STORED == 1> sum(v[k][0]);
#pragma unroll
                for (int h = 1; h < N; ++h) sum.add(v[k][h]);
                u32x4 x = sum.value();
                if constexpr (FORM::kLarge) cu_pause(pauses, x);
#pragma unroll
                for (int i = 0; i < STORED; ++i) at.template store<FORM::kStores>(i, base + k * kStep, lane, x);
            }
        });
        return;
    }
    typename Row::Bytes off;
    if (tile > tiles || !row.end_element(DT == DT_F32 ? 4u : 2u, off)) return;
    uint32_t v[N];
#pragma unroll
    for (int h = 0; h < N; ++h) v[h] = at.template load_element<DT>(h, off);
    uint32_t x = v[0];
#pragma unroll
    for (int h = 1; h < N; ++h) x = add_rn<DT>(v[h], x);
#pragma unroll
    for (int i = 0; i < STORED; ++i) at.template store_element<DT>(i, off, x);
}
template <int DT, int N, bool EVERYWHERE, typename FORM, bool SPLIT>
__global__ void __launch_bounds__(FORM::kThreads) cu_ring_sum_kernel(u64x4 numbers, u32x2 counts, const CuTables<N, SPLIT> a) {
    const CuShape s(numbers, counts);
    constexpr uint32_t kSize = DT == DT_F32 ? 4u : 2u;
    const CuPlace place(FORM::kLarge, s.part);
    const uint32_t tile = place.tile, p = place.pipe;
    const uint32_t root = s.starts >> (3u * p) & 7u;
    constexpr int kStored = EVERYWHERE ? N : 1, kOut = SPLIT ? N : 0;
    CuByTable<N, kStored> at;
    at.row_off = (uint64_t)p * s.row_stride;
    // (all of them asked for before the first is waited for: large sums to one place, whose
    // few wavefronts do not hide a second wait: 8 ranks, 0.99 at 110 - 180 MiB touched)
#pragma unroll
    for (int i = 0; i < kStored; ++i) at.to[i] = reinterpret_cast<uint8_t*>(a.rank[kOut + (EVERYWHERE ? (uint32_t)i : root)]);
    cu_around(a.rank, root, at.from);
    if constexpr (EVERYWHERE || SPLIT) cu_here(at.to);
    else at.to[0] = const_cast<uint8_t*>(at.from[0]);
    const CuRow<FORM> row(s.row_bytes, s.short_bytes, s.full, p, at.to[0] + at.row_off, kSize);
    cu_count_if_aborted<FORM::kThreads>(a.status);
    cu_sum_row<DT, N, kStored>(row, tile, s.tiles, s.part, at);
}
template <int DT, int N, bool EVERYWHERE, typename FORM, typename... MORE>
__global__ void __launch_bounds__(FORM::kThreads) cu_near_sum_kernel(u32x8 rows, u32x4 words, MORE... more) {
    const CuNear a(FORM::kLarge, rows, words, more...);
    const CuPlace place(FORM::kLarge, a.part);
    const uint32_t p = place.pipe;
    const CuByDistance<N, 0> at(a, a.root(p), p * a.row_stride);
    const auto row = a.template row<FORM>(p, at.stored(), DT == DT_F32 ? 4u : 2u);
    cu_count_if_aborted<FORM::kThreads>(a.status);
    cu_sum_row<DT, N, EVERYWHERE ? N : 1>(row, place.tile, a.tiles, a.part, at);
}

// A row from one place to COPIES others.
template <int COPIES, typename FORM, bool WIDE, typename PLACES>
__device__ __forceinline__ void cu_copy_row(const CuRow<FORM, WIDE>& row, uint32_t tile, uint32_t tiles, uint32_t pauses, const PLACES& at) {
    using Row = CuRow<FORM, WIDE>;
    if (__builtin_expect(tile < tiles, 1)) {
        const uint32_t lane = threadIdx.x * 16u;
        row.tiles(tile, tiles, [&](typename Row::Offset base, auto count) MINT_INLINE_LAMBDA {
            constexpr int kCount = decltype(count)::value, kStep = FORM::kThreads * 16;
            u32x4 x[kCount];
#pragma unroll
            for (int k = 0; k < kCount; ++k) x[k] = at.template load<FORM::kStream>(0, base + k * kStep, lane);
            if constexpr (FORM::kLarge && COPIES == 1) cu_pause(pauses, x[0]);
#pragma unroll
            for (int k = 0; k < kCount; ++k)
#pragma unroll
                for (int i = 0; i < COPIES; ++i) at.template store<FORM::kStores>(i, base + k * kStep, lane, x[k]);
        });
        return;
    }
    typename Row::Bytes off;
    if (tile > tiles || !row.end_element(1u, off)) return;
    const uint32_t x = at.template load_element<DT_BYTES>(0, off);
#pragma unroll
    for (int i = 0; i < COPIES; ++i) at.template store_element<DT_BYTES>(i, off, x);
}

// Rings that copy: N ranks, the root's row to every other one (broadcast,
// allgather).  A route is a ring of its two ends (sendrecv).
template <int N, typename FORM, bool SPLIT>
__global__ void __launch_bounds__(FORM::kThreads) cu_ring_copy_kernel(u64x4 numbers, u32x2 counts, const CuTables<N, SPLIT> a) {
    const CuShape s(numbers, counts);
    const CuPlace place(FORM::kLarge, s.part);
    const uint32_t p = place.pipe;
    const uint32_t root = s.starts >> (3u * p) & 7u;
    constexpr uint32_t kOut = SPLIT ? N : 0;
    CuByTable<1, N - 1> at;
    at.row_off = (uint64_t)p * s.row_stride;
    at.from[0] = reinterpret_cast<const uint8_t*>(a.rank[root]);
    uint8_t* all[N];
#pragma unroll
    for (int k = 0; k < N; ++k) all[k] = reinterpret_cast<uint8_t*>(a.rank[kOut + k]);
    cu_here(at.from);
    cu_here(all);
#pragma unroll
    for (int k = 0; k < N - 1; ++k) at.to[k] = (uint32_t)k < root ? all[k] : all[k + 1];
    const CuRow<FORM> row(s.row_bytes, s.short_bytes, s.full, p, at.to[0] + at.row_off, 1u);
    cu_count_if_aborted<FORM::kThreads>(a.status);
    cu_copy_row<N - 1>(row, place.tile, s.tiles, s.part, at);
}
template <int N, typename FORM, typename... MORE>
__global__ void __launch_bounds__(FORM::kThreads) cu_near_copy_kernel(u32x8 rows, u32x4 words, MORE... more) {
    const CuNear a(FORM::kLarge, rows, words, more...);
    const CuPlace place(FORM::kLarge, a.part);
    const uint32_t p = place.pipe;
    const CuByDistance<N, 1> at(a, a.root(p), p * a.row_stride);
    const auto row = a.template row<FORM>(p, at.stored(), 1u);
    cu_count_if_aborted<FORM::kThreads>(a.status);
    cu_copy_row<N - 1>(row, place.tile, a.tiles, a.part, at);
}

// The addresses of an alltoall, N to load from and N to store to.  T = uint32_t
// where they lie whole multiples of 256 bytes from the lowest, as allocations do:
// their distances from it in those units, which keeps a launch below 112 bytes of
// arguments (2.7 us for the host; with 64-bit ones, 168 bytes, 3.4 - 3.5).
template <typename T>
struct CuPairs {
    T rank[2 * kMaxRanks];
};
constexpr int kCuNearShift = 8;
static_assert(5 * 8 + sizeof(CuPairs<uint32_t>) <= 112, "arguments of an alltoall's launch");

// Row `destination` of the source goes to row `source` of the destination.
template <typename FORM>
__device__ __forceinline__ void cu_alltoall_row(uint64_t from, uint64_t to, uint64_t row_bytes, uint64_t row_stride, uint32_t tiles,
                                                uint32_t part, const CuPlace& place, uint64_t* status) {
    CuByTable<1, 1> places;
    places.from[0] = reinterpret_cast<const uint8_t*>(from) + (uint64_t)place.pipe * row_stride;
    places.to[0] = reinterpret_cast<uint8_t*>(to) + (uint64_t)blockIdx.z * row_stride;
    places.row_off = 0;
    cu_count_if_aborted<FORM::kThreads>(status);
    cu_copy_row<1>(CuRow<FORM>(row_bytes, 0u, kMaxRanks, place.pipe, places.to[0], 1u), place.tile, tiles, part, places);
}
// `numbers`: row_bytes, row_stride, the lowest address, the status block.
template <typename FORM, typename T>
__global__ void __launch_bounds__(FORM::kThreads) cu_alltoall_kernel(u64x4 numbers, u32x2 counts, const CuPairs<T> a) {
    const uint64_t lowest = numbers.z;
    const CuPlace place(FORM::kLarge, counts.y);
    T load = a.rank[blockIdx.z], store = a.rank[kMaxRanks + place.pipe];
    asm volatile("" : "+s"(load), "+s"(store));                 // (see cu_here)
    const auto at = [&](T x) MINT_INLINE_LAMBDA { return sizeof(T) == 4 ? lowest + ((uint64_t)x << kCuNearShift) : (uint64_t)x; };
    cu_alltoall_row<FORM>(at(load), at(store), numbers.x, numbers.y, counts.x, counts.y, place, reinterpret_cast<uint64_t*>(numbers.w));
}
// Up to four ranks, whose rows follow each other without gaps: all that the loads wait for in the
// 14 words that come in registers (CuNear); the selects of a block's two distances take no longer than one to a
// table's entry. Over tables, the same buffers again / three sets in turn:
//   touched MiB      20             30             45             64             90            150
//   2 ranks     0.95 / 0.95    0.97 / 0.97    0.99 / 0.97    0.97 / 0.98    0.98 / 0.98   0.99 / 0.99
//   3           0.99 / 0.95    0.98 / 0.95    0.99 / 0.97    0.97 / 0.98    0.98 / 0.98   0.99 / 0.99
//   4           0.97 / 0.93    0.95 / 0.96    0.96 / 0.97    0.98 / 0.98    0.98 / 0.98   0.99 / 0.99
// (4 ranks of 30 MiB, three sets, 5.36 -> 5.13 us, 6.1 TB/s; 64 MiB 10.22 -> 9.99; 90 MiB 13.8 -> 13.6).  Up to 12 MiB the host's launch is
// what a call takes, 0.985 - 1.016 with a scatter of 5 %; from 200 MiB on it is the large form, by tables.  More ranks: 16 distances of 20
// bits, in halves and fours, fit as well, but finding two of them takes
// about what the table does (5 and 6 ranks 0.98 - 1.02, 7 and 8 ranks 0.98 - 1.01).
//   rows    lowest address (two words), row_bytes, tiles | part << cu_near_part_bit; what ranks 0 - 3 load from
//   stored  what they store to
constexpr uint32_t kCuNearPairs = 4;
template <typename FORM>
__global__ void __launch_bounds__(FORM::kThreads) cu_near_alltoall_kernel(u32x8 rows, u32x4 stored, uint64_t* status) {
    static_assert(!FORM::kLarge, "rows of 32 bits, tiles and their part in a word");
    constexpr uint32_t kBit = cu_near_part_bit(false);
    const uint64_t lowest = (uint64_t)rows[1] << 32 | rows[0];
    const uint32_t tiles = rows[3] & ((1u << kBit) - 1u), part = rows[3] >> kBit;
    const CuPlace place(false, part);
    const auto at = [&](uint32_t r, uint32_t a, uint32_t b, uint32_t c, uint32_t d) MINT_INLINE_LAMBDA {
        const uint32_t low = r & 1u ? b : a, high = r & 1u ? d : c;
        return lowest + ((uint64_t)(r & 2u ? high : low) << kCuNearShift);
    };
    cu_alltoall_row<FORM>(at(blockIdx.z, rows[4], rows[5], rows[6], rows[7]), at(place.pipe, stored.x, stored.y, stored.z, stored.w),
                          rows[2], rows[2], tiles, part, place, status);
}

}  // namespace mint
