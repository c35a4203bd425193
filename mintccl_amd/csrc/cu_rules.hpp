// How many wavefronts of a launch inside compute units (cu_ring.hpp) a compute unit is to hold, and how long
// they wait before they store: functions of what is moved alone.  Host code without a line of HIP,
// so that any C++ compiler can say what they give.
#pragma once
#include <cstdint>

#include "../../include/mintccl.h"

namespace mint {

constexpr int kCuMostWaves = 32;               // that a compute unit holds
constexpr uint32_t kCuLds = 160u << 10;        // bytes of LDS of a compute unit, handed out in units of
constexpr uint32_t kCuLdsUnit = 1280;
// The LDS that a block of `threads` asks for so that a compute unit holds `waves` wavefronts of them, one
// block at least.
constexpr uint32_t cu_lds_share(int waves, int threads) {
    if (waves >= kCuMostWaves) return 0;
    const int blocks = waves * 64 / threads;
    return kCuLds / (uint32_t)(blocks > 1 ? blocks : 1) / kCuLdsUnit * kCuLdsUnit;
}
constexpr bool cu_adds(int op) { return op == MINT_OP_REDUCE || op == MINT_OP_REDUCESCATTER || op == MINT_OP_ALLREDUCE; }

// The wavefronts that a compute unit is to hold of the large form of a launch
// inside compute units (cu_ring.hpp; one copy of a row: all 32).  Some 64 KiB
// of rows on their way to or from a compute unit keep HBM busy: fewer
// wavefronts leave it idle, more only scatter its accesses.  Each holds a KiB of
// N rows to be added, of a row that goes to N - 1 others, or (allreduce) of N rows
// and then N results.  One or two off is 1 - 3 % slower, twice as many 5 - 20 %.
// Launches by distances (CuNear), whose wavefronts are sooner at their loads, over
// the number that launches by tables want, three sets of buffers in turn (in no cache alike):
//   sums, one fewer: 4 ranks 0.98 from 530 MiB on (290 1.02, 430 0.99); 5 ranks 1.02 at 290 - 430, 0.99
//     beyond; 7 ranks 0.985 - 0.99 throughout; 6 and 8 ranks 1.00 - 1.04
//   (a sum of two ranks, 20 for 18, by cu_pauses: see there; an allreduce of four, f16 and f32, 9 and a wait of 768 clocks for 8 and
//     none, one process: 0.976 - 1.003, geometric mean 0.995)
// Copies of seven and eight ranks beyond 72 MiB copied: 10 (72 MiB 88.1 with 8, 87.7 with 10; 128 MiB 178 / 174).
// Copies with fewer wavefronts than these (8 / 8 / 5 / 6 of 5 / 6 / 7 / 8 ranks up to 72 MiB copied) are ahead on
// buffers that have just been used and behind where 1.3 GB and more lie between two uses, as with first uses:
// an access waits for its address's translation too then, and more of them have to be under
// way.  Over these, geometric means, the same buffers again / three sets in turn / 3.5 GB between two uses:
//   touched MiB      90 - 150               180 - 260              310 - 570
//   5 ranks    0.92 / 0.98 / 1.18    0.99 / 0.98 / 1.19    0.98 / 0.98 / 1.20
//   6          0.93 / 0.98 / 1.10    0.96 / 0.97 / 1.11    0.99 / 0.98 / 1.12
//   7          0.95 / 0.99 / 1.20    0.96 / 0.97 / 1.21    0.97 / 0.98 / 1.22
//   8          1.00 / 1.01 / 1.07    0.97 / 1.00 / 1.08    1.00 / 1.00 / 1.10
constexpr int cu_waves(int op, int dtype, int ranks, bool vast, uint64_t copied) {
    const uint64_t touched = copied * (uint64_t)ranks;
    if (op == MINT_OP_ALLREDUCE) return (26 + ranks - 1) / ranks + 1 + (ranks == 4 && dtype != MINT_BF16);
    if (cu_adds(op)) {
        if (ranks == 2) return 20;
        if (ranks == 4) return touched <= (320ull << 20) ? 12 : 11;
        if (ranks == 5) return touched <= (480ull << 20) ? 11 : 10;
        // (7 ranks, 10 for 9, the same buffers again / three sets in turn / 700 MiB between two uses: 104 MiB 0.97 / 0.985 / 0.985,
        // 130 MiB 0.975 / 0.995 / 0.995, 150 MiB 0.98 / 0.995 / 0.995, 180 MiB 0.985 / 1.005 / 1.01)
        if (ranks == 7 && touched <= (160ull << 20)) return 10;
        return ranks == 6 ? 10 : 24 / ranks + 6;
    }
    if (vast) return ranks == 6 ? 5 : 4;
    return ranks < 7 ? 24 - 2 * ranks : copied <= (72ull << 20) ? 8 : 10;
}

// ... of the form between.  4 ranks, over 32, the same buffers again / three sets in turn / 700 MiB between two uses: 105 - 125 MiB 18
// 1.00 / 0.985 / 0.98 (16: 1.02 / 0.975 / 0.975), 150 MiB 22 0.99 / 0.995 / 0.99 (18: 1.03 / 0.99 / 0.99), 170 - 205 MiB 16
// 0.975 / 0.97 / 0.97 (18: 0.99).  In one process over 18 throughout: 130 - 165 MiB 0.99 / 1.007 / 1.006 (22 is there for the same buffers
// again, 0.95 - 0.995 at 150 MiB, where 18 is behind 32), 165 - 208 MiB 0.98 / 0.98 / 0.99; 2 ranks 24 1.02 - 1.05; 3 ranks 24 0.99 - 1.00.  5 and 6 ranks: kCuMidRanks.
constexpr int cu_mid_waves(int ranks, uint64_t touched) {
    if (ranks == 4) return touched <= (130ull << 20) ? 18 : touched <= (165ull << 20) ? 22 : 16;
    return ranks < 4 ? kCuMostWaves : 14;
}

// ... and of the small form of an allreduce, which stores as many rows as it loads, once it touches about as much as the L2s hold.
// Over all 32, f16 and bf16, the same buffers again / three sets in turn / 700 MiB between two uses:
//   touched MiB        26                 36                 48                 60                 72                 98
//   2 ranks, 20  0.97 / 0.97 / 0.97  0.98 / 0.98 / 0.96  0.99 / 0.99 / 0.97  0.99 / 0.99 / 0.96  0.99 / 0.99 / 0.97  0.99 / 0.99 / 0.97
//   3, 16        0.98 / 0.98 / 0.98  1.00 / 1.00 / 0.99  0.99 / 0.99 / 0.98  1.00 / 0.99 / 0.97  0.99 / 0.99 / 0.97  0.98 / 0.97 / 0.97
//   4, 12        0.99 / 0.98 / 0.97  0.97 / 0.97 / 0.99  0.98 / 0.98 / 0.97  0.98 / 0.98 / 0.98  0.98 / 0.98 / 0.98  0.98 / 0.99 / 0.97
//   5, 8         0.98 / 0.98 / 0.97  0.98 / 0.97 / 0.98  0.98 / 0.98 / 0.97  0.98 / 0.97 / 0.97  0.98 / 0.98 / 0.97  0.98 / 1.00 / 0.98
//   6, 8         1.01 / 1.01 / 0.99  0.98 / 0.98 / 0.99  0.98 / 0.98 / 0.98  0.98 / 0.98 / 0.98  0.98 / 0.98 / 0.99  0.98 / 1.00 / 0.99
//   7, 8         1.00 / 0.99 / 1.00  0.99 / 0.99 / 0.98  0.99 / 0.99 / 0.98  0.99 / 0.99 / 0.98  0.99 / 0.96 / 0.99  1.00 / 1.00 / 0.99
// (3 and 4 ranks of bf16 at 25 MiB 1.01 - 1.03 / 1.00 - 1.01 / 0.98.)  Up to 20 MiB as fast or slower; 8 ranks 1.00 - 1.05. Sums to one place 1.00 - 1.1, copies 0.96 - 1.08 by their size.
constexpr int cu_small_waves(int op, int ranks, uint64_t touched) {
    const uint64_t least = ranks == 2 || ranks == 5 ? 24 : ranks <= 4 ? 28 : 32;
    if (op != MINT_OP_ALLREDUCE || ranks == 8 || touched < least << 20) return kCuMostWaves;
    return ranks == 2 ? 20 : ranks == 3 ? 16 : ranks == 4 ? 12 : 8;
}

// Times 256 clocks that a wavefront of the large form, its rows there and added, waits
// before it stores (cu_pause).  It is the spread of the accesses that this holds down, like a wavefront less on
// the compute unit does (cu_waves) but in smaller steps, and the stores: as far as can be told, HBM loses time where
// they come one by one between the loads.  Additions of bf16, which are conversions too, are a part of the wait.  Time over
// that without, in thousandths, f16 and f32 / bf16, reduce-scatter and reduce, up to 200 MiB the same buffers again
// and three sets in turn, beyond three sets:
//   touched MiB       180 - 200          300          500 - 700         1000            2000
//   2 ranks (20 wf.)      -           968 / 987      965 / 988       968 / 978       971 / 985
//   3                     -           971 / -        976 / -         976 / -         967 / -
//   4                     -           957 / -        981 / -         988 / -         956 / -
//   5                938 - 972 / 987  963 / 991      973 / 992       979 / 986       976 / 988
//   6                961 - 984 / 993  973 / 984      977 / 990       995 / 1003      993 / 997
//   7                962 - 989 / 992  981 / 1000     982 / 993      1004 / 1005     1013 / 1006
//   8                990 - 1037 / 1010  984 / 1000   977 / 980       976 / 975      1003 / 996
// Two more are 1 - 5 % slower.  Allreduce, f16 and f32, geometric means of 102 - 2500 MiB (largest), the same buffers again / three
// sets in turn / 3.5 GB between two uses: 8 ranks (bf16 too) 993 (1006) / 992 (1006) / 991 (1003), 7 ranks 996 (1007) / 995 (1003) / 993, 6 ranks
// 998 (1010) / 994 / 990, 5 ranks 997 (1010) / 996 (1005) / 992, 4 ranks (nine wavefronts) 991 / 992 / 989; the same build on both
// sides 996 - 1003.  bf16 of 7 ranks up to 150 MiB, 512 clocks: 1002 (1010) / 1001 (1007) / 998, no gain; 2 and 3 ranks lose by it.
// One copy: sendrecv 954 - 997 from 200 MiB on, alltoall 1000 - 1009 at 200 - 300, 991 at 1000, 985 at 2000.
// Several copies of a row lose 3 % and more: their stores are most of what there is.
constexpr uint32_t cu_pauses(int op, int dtype, int ranks, uint64_t touched) {
    const auto upto = [&](uint64_t mib) { return touched <= mib << 20; };
    const bool bf16 = dtype == MINT_BF16;
    if (op == MINT_OP_ALLREDUCE) {
        if (ranks == 8) return bf16 ? 3 : 4;
        return ranks < 4 || bf16 ? 0 : ranks == 4 ? 3 : 2;
    }
    if (cu_adds(op)) {
        switch (ranks) {
            case 8: return bf16 ? (upto(400) ? 0 : 3) : upto(240) || !upto(1500) ? 0 : 4;
            case 7: return upto(160) || !upto(800) ? 0 : bf16 ? 1 : 3;
            case 6:
            case 5: return bf16 ? 1 : 3;
            case 4:
            case 3: return bf16 ? 0 : 2;
            default: return 3;
        }
    }
    if (op == MINT_OP_ALLTOALL) return upto(400) ? 0 : 2;
    return ranks == 2 ? 2 : 0;
}

}  // namespace mint
