// Rings inside a compute unit: the ring collectives of ring.hpp with every
// position of a channel in ONE thread block and the hops between them in LDS.
//
// The walks of ring.hpp put neighbouring positions on different compute units
// and their staging into the L2 of an XCD.  A hop then costs a 1 KiB store and
// a 1 KiB load through the L2 beside the rows from HBM, and a compute unit
// keeps only some 130 requests in flight: an 8-rank reduce-scatter spends half
// of its time on staging.  Virtual ranks share one GPU, so a channel's whole
// ring fits one compute unit: wavefront h of the block is position h (the rank
// `h` places after the pipeline's root), it loads its own rank's row from HBM
// ahead of time, takes the block its predecessor left in LDS, adds or copies,
// and leaves the result for its successor.  What crosses the memory system is
// each row once; LDS carries 2 KiB per hop and KiB of row, an eighth of its rate.
//
// The wire between two positions: NS slots of U KiB in LDS, and two words,
//   head   steps the sender has put into the slots   (sender writes)
//   tail   steps the receiver has taken out          (receiver writes)
// the pair of the Simple protocol (post / wait, protocol.py:161-189).  LDS
// executes a wavefront's operations in issue order, so a `head` stored behind
// the data is seen behind the data: what LL128's flag inside every line is for
// holds by itself, and both protocols move whole 1 KiB blocks here.  There is
// no epoch, no staging memory and no seat to claim: the words start at zero in
// every block, all positions of a channel are resident together because they
// are one block, and a grid of any size drains.  Waits stay bounded and report
// like those of ring.hpp.
#pragma once
#include "ring.hpp"

namespace mint {

// One launch.  The ranks' buffers come in the order of the ring (or route), so
// that position h of a pipeline that starts at index i works for index
// (i + h) % len of these tables.
struct CuRingArgs {
    uint64_t input[kMaxRanks], output[kMaxRanks];
    uint64_t starts;               // byte p: index in the ring of pipeline p's root
    uint64_t row_bytes, row_stride;
    uint64_t total_bytes;          // 0, or clip row p to total_bytes - p * row_stride
    uint64_t* status;
    uint32_t op, pipes, len, hops;
    uint32_t channels;             // per pipeline
    uint32_t spin_budget;
};

// Row p in whole 1 KiB blocks, dealt in units of `unit`: unit i belongs to
// channel i % channels, which walks its units in steps.  The bytes behind the
// last whole block are a step of their own of the channel that comes next.
struct CuWalk {
    uint32_t steps;          // units of this channel
    uint32_t nfull;          // whole blocks of the row
    bool tail;               // this channel moves the bytes behind them
    uint64_t row_bytes;
};
__host__ __device__ __forceinline__ CuWalk cu_walk_of(const CuRingArgs& a, uint32_t p, uint32_t c,
                                                      uint32_t unit) {
    CuWalk k;
    k.row_bytes = a.row_bytes;
    if (a.total_bytes) {
        const uint64_t off = (uint64_t)p * a.row_stride;
        const uint64_t left = a.total_bytes > off ? a.total_bytes - off : 0;
        k.row_bytes = left < a.row_bytes ? left : a.row_bytes;
    }
    k.nfull = (uint32_t)(k.row_bytes / kBlockRawSimple);
    const uint32_t units = (k.nfull + unit - 1) / unit;
    k.steps = units > c ? (units - 1 - c) / a.channels + 1 : 0;
    k.tail = k.row_bytes % kBlockRawSimple != 0 && units % a.channels == c;
    return k;
}

// The words of a channel, in LDS in front of the slots: head and tail of every hop.
constexpr int kCuMaxHops = 2 * kMaxRanks - 2;
constexpr uint32_t kCuWordBytes = 128;
static_assert(2 * kCuMaxHops * 4 <= (int)kCuWordBytes, "head and tail of every hop");

// What a position does, in flags that are compile-time constants of its walk.
template <bool LOAD, bool RECV, bool REDUCE, bool SAVE, bool SEND>
struct CuRole {
    static constexpr bool load = LOAD, recv = RECV, reduce = REDUCE, save = SAVE, send = SEND;
};

// Polls `word` until it has reached `need` or `patience` further polls have
// gone by; `seen` comes back as what the last poll saw.
__device__ __forceinline__ void cu_spin(MINT_LDS const uint32_t* word, uint32_t need, uint32_t patience,
                                        uint32_t& seen) {
    uint32_t v, gap;
    asm volatile(
        "1:\n\t"
        "ds_read_b32 %[v], %[word]\n\t"
        "s_waitcnt lgkmcnt(0)\n\t"
        "v_readfirstlane_b32 %[seen], %[v]\n\t"
        "s_sub_i32 %[gap], %[seen], %[need]\n\t"
        "s_cmp_ge_i32 %[gap], 0\n\t"
        "s_cbranch_scc1 2f\n\t"
        "s_sub_u32 %[left], %[left], 1\n\t"
        "s_cbranch_scc1 2f\n\t"
        "s_sleep 1\n\t"
        "s_branch 1b\n"
        "2:"
        : [v] "=&v"(v), [seen] "=&s"(seen), [gap] "=&s"(gap), [left] "+s"(patience)
        : [word] "v"(word), [need] "s"(need)
        : "memory", "scc");
}

template <int DT, int U, int NS, int D, typename Role>
__device__ __forceinline__ void cu_walk(const CuRingArgs& a, const uint32_t p, const uint32_t h,
                                        const uint32_t c, const uint8_t* in_row, uint8_t* out_row,
                                        MINT_LDS uint8_t* lds, Role) {
    static_assert((NS & (NS - 1)) == 0 && D == 4, "masks; the loop below is unrolled by the depth");
    constexpr uint32_t kSlot = (uint32_t)U * kBlockRawSimple, kHop = (uint32_t)NS * kSlot;
    const uint32_t lane_off = (uint32_t)lane_id() * 16u;
    const CuWalk k = cu_walk_of(a, p, c, (uint32_t)U);
    MINT_LDS uint32_t* const head = reinterpret_cast<MINT_LDS uint32_t*>(lds);
    MINT_LDS uint32_t* const tail = head + kCuMaxHops;
    MINT_LDS uint8_t* const slots = lds + kCuWordBytes;
    MINT_LDS uint8_t* const rx = slots + (h - 1u) * kHop + lane_off;
    MINT_LDS uint8_t* const tx = slots + h * kHop + lane_off;
    const uint32_t C = a.channels, last = k.nfull - 1u;

    // Own rows, D steps ahead.  Block numbers are clamped to the last whole
    // block, so that every step issues the same loads and the wait for the
    // oldest leaves the others in flight.  The walk is whole rounds of D steps
    // with one way out (the compiler sets each wait from the path with the
    // fewest younger loads, and an exit in the middle of a round would be
    // such a path): what the steps leave over D comes first, so buffer j
    // starts with step (j + rest) % D.
    u32x4 v[D][U];
    auto fetch = [&](uint32_t s, u32x4 (&x)[U]) MINT_INLINE_LAMBDA {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint32_t g = (s * C + c) * (uint32_t)U + (uint32_t)u;
            g = g < last ? g : last;
            x[u] = ld128_row(in_row + (uint64_t)g * kBlockRawSimple + lane_off);
        }
    };
    const uint32_t rest = k.steps % (uint32_t)D;
    if (Role::load && k.steps) {
#pragma unroll
        for (int d = 0; d < D; ++d) fetch(((uint32_t)d + rest) % (uint32_t)D, v[d]);
    }
    // The words are cleared while the first rows are on their way; the barrier
    // must not wait for those.
    if (threadIdx.x < kCuWordBytes / 4) head[threadIdx.x] = 0u;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // wait_ll128 (protocol.py:161-180) on either word.  A wait that runs out
    // marks the walk as failed and lets it go on without waiting any further:
    // the outputs are unspecified from there on, every access stays where it
    // was, the neighbours see their words move and the grid drains.  (Written
    // as one statement, with no way out of the walk behind it, so that the
    // compiler keeps exact count of the loads in flight around it.)
    uint32_t head_seen = 0, tail_seen = 0, patience = a.spin_budget, failed_at = ~0u;
    auto wait_for = [&](MINT_LDS uint32_t* word, uint32_t need, uint32_t& seen, uint32_t s) MINT_INLINE_LAMBDA {
        if ((int32_t)(seen - need) >= 0) return;
        cu_spin(word, need, patience, seen);
        if ((int32_t)(seen - need) < 0) {
            failed_at = failed_at < s ? failed_at : s;
            patience = 0;
        }
    };
    // One step between this position's neighbours: take the blocks out of the
    // predecessor's slot, combine them with `own`, leave them for the successor.
    auto pass_on = [&](uint32_t s, const u32x4 (&own)[U], u32x4 (&x)[U]) MINT_INLINE_LAMBDA {
        const uint32_t slot = (s & (uint32_t)(NS - 1)) * kSlot;
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = own[u];
        if (Role::recv) {
            wait_for(head + (h - 1u), s + 1u, head_seen, s);
            compiler_fence();
            u32x4 r[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                r[u] = *reinterpret_cast<MINT_LDS const u32x4*>(rx + slot + (uint32_t)u * kBlockRawSimple);
            // post_ll128 (protocol.py:183-189): executed behind the reads
            compiler_fence();
            lds_set(tail + (h - 1u), s + 1u);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if constexpr (DT != DT_BYTES) x[u] = Role::reduce ? ll_comp<DT>(x[u], r[u]) : r[u];
                else x[u] = r[u];
            }
        }
        if (Role::send) {
            wait_for(tail + h, s + 1u - (uint32_t)NS, tail_seen, s);
            compiler_fence();
#pragma unroll
            for (int u = 0; u < U; ++u)
                *reinterpret_cast<MINT_LDS u32x4*>(tx + slot + (uint32_t)u * kBlockRawSimple) = x[u];
            compiler_fence();
            lds_set(head + h, s + 1u);
        }
    };
    uint32_t s = 0;
    auto step = [&](auto phase) MINT_INLINE_LAMBDA {
        constexpr int B = decltype(phase)::value;
        u32x4 x[U];
        pass_on(s, v[B], x);
        if (Role::save) {
            const uint32_t g = (s * C + c) * (uint32_t)U;
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (U == 1 || g + (uint32_t)u < k.nfull)
                    st128_row(out_row + (uint64_t)(g + (uint32_t)u) * kBlockRawSimple + lane_off, x[u]);
        }
        if (Role::load) {
            compiler_fence();
            fetch(s + (uint32_t)D, v[B]);
        }
        ++s;
    };
    if (rest >= 3u) step(std::integral_constant<int, 1>{});
    if (rest >= 2u) step(std::integral_constant<int, 2>{});
    if (rest >= 1u) step(std::integral_constant<int, 3>{});
    while (s != k.steps) {
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
    }
    if (k.tail) {
        // fewer than 1 KiB, byte by byte where a lane's 16 are not all there
        u32x4 own[U], x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) own[u] = u32x4{0u, 0u, 0u, 0u};
        const uint64_t off = (uint64_t)k.nfull * kBlockRawSimple + lane_off;
        if (Role::load) own[0] = load_guarded(in_row, off, 16u, k.row_bytes);
        pass_on(k.steps, own, x);
        if (Role::save) store_guarded(out_row, off, 16u, k.row_bytes, x[0]);
    }
    if (failed_at != ~0u) report_timeout(a.status, (int)p, (int)h, (int)c, failed_at);
    // a launch that finds the abort flag set is counted, as in take_seat
    if (!Role::recv) count_launch_if_aborted(a.status, (int)h);
}

// One thread block per channel: wavefront h is position h (the roles: role_of).
template <int DT, int U, int NS, int D>
__global__ void __launch_bounds__((2 * kMaxRanks - 1) * 64) cu_ring_kernel(const CuRingArgs a) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    MINT_LDS uint8_t* lds = (MINT_LDS uint8_t*)lds_raw;
    const uint32_t h = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)wave_in_block());
    const uint32_t c = blockIdx.x / a.pipes, p = blockIdx.x - c * a.pipes;
    uint32_t row_in = p, row_out = p, idx;
    if (a.op == OP_ALLTOALL) {
        // pipeline source * len + destination
        row_out = p / a.len;
        row_in = p - row_out * a.len;
        idx = h == 0u ? row_out : row_in;
    } else {
        idx = (uint32_t)(a.starts >> (8u * p)) & 0xFFu;
        idx += h;
        while (idx >= a.len) idx -= a.len;
    }
    const uint8_t* in_row = reinterpret_cast<const uint8_t*>(a.input[idx]) + (uint64_t)row_in * a.row_stride;
    uint8_t* out_row = reinterpret_cast<uint8_t*>(a.output[idx]) + (uint64_t)row_out * a.row_stride;
    const bool sink = h == a.hops, allreduce = a.op == OP_ALLREDUCE;
    if (h == 0u) {
        cu_walk<DT, U, NS, D>(a, p, h, c, in_row, out_row, lds, CuRole<true, false, false, false, true>{});
        return;
    }
    if constexpr (DT != DT_BYTES) {
        if (allreduce ? h < a.len : !sink) {
            if (allreduce && h == a.len - 1u)
                cu_walk<DT, U, NS, D>(a, p, h, c, in_row, out_row, lds, CuRole<true, true, true, true, true>{});
            else
                cu_walk<DT, U, NS, D>(a, p, h, c, in_row, out_row, lds, CuRole<true, true, true, false, true>{});
            return;
        }
    }
    if (sink)
        cu_walk<DT, U, NS, D>(a, p, h, c, in_row, out_row, lds, CuRole<false, true, false, true, false>{});
    else if (a.op == OP_SENDRECV)
        cu_walk<DT, U, NS, D>(a, p, h, c, in_row, out_row, lds, CuRole<false, true, false, false, true>{});
    else
        cu_walk<DT, U, NS, D>(a, p, h, c, in_row, out_row, lds, CuRole<false, true, false, true, true>{});
}

}  // namespace mint
