// The kernels of rings inside compute units (cu_ring.hpp) and their launcher.
#include <algorithm>

#include "ring_launch.hpp"

namespace mint {
namespace {

// `rows`: pipelines, alltoall: destinations
dim3 grid_of(const Plan& plan, uint32_t rows, uint32_t sources) {
    const CuRingArgs& a = plan.cu_args;
    const bool by_row = plan.cu_large || a.shape.part;
    return dim3(by_row ? a.blocks : rows, by_row ? rows : a.blocks, sources);
}

template <auto KERNEL, int N, bool SPLIT>
int launch_as(const Plan& plan, hipStream_t stream) {
    const CuRingArgs& a = plan.cu_args;
    const CuShape& s = a.shape;
    CuTables<N, SPLIT> tables = {};
    for (uint32_t i = 0; i < a.len; ++i) {
        tables.rank[i] = SPLIT || a.input[i] ? a.input[i] : a.output[i];
        if (SPLIT) tables.rank[N + i] = a.output[i];
    }
    tables.status = a.status;
    u64x4 numbers;
    s.numbers(numbers);
    return Launch<KERNEL>::go(grid_of(plan, a.pipes, 1), (unsigned)plan.threads, (unsigned)plan.cu_lds, stream,
                              numbers, u32x2{s.tiles, s.part}, tables);
}

// (in place only in the small form: to the large one the host's time is nothing)
template <int DT, int N, bool EVERYWHERE>
int launch_sum(const Plan& plan, hipStream_t stream) {
    if constexpr (N >= kCuStreamRanks && !EVERYWHERE)
        if (plan.cu_far)
            return launch_as<&cu_ring_sum_kernel<DT, N, EVERYWHERE, CuLargeSumStreamed, true>, N, true>(plan, stream);
    if constexpr (N <= kCuMidRanks && !EVERYWHERE)
        if (plan.cu_mid) return launch_as<&cu_ring_sum_kernel<DT, N, EVERYWHERE, CuMidSum<N>, true>, N, true>(plan, stream);
    using Large = std::conditional_t<EVERYWHERE, CuLargeSumEverywhere, CuLargeSum>;
    if (plan.cu_large) return launch_as<&cu_ring_sum_kernel<DT, N, EVERYWHERE, Large, true>, N, true>(plan, stream);
    const auto small = [&](auto form) {
        using Small = decltype(form);
        if (plan.cu_args.split)
            return launch_as<&cu_ring_sum_kernel<DT, N, EVERYWHERE, Small, true>, N, true>(plan, stream);
        return launch_as<&cu_ring_sum_kernel<DT, N, EVERYWHERE, Small, false>, N, false>(plan, stream);
    };
    if constexpr (EVERYWHERE || N <= kCuThroughRanks) return small(CuSmall<true>{});
    else return plan.cu_through ? small(CuSmallSum<true>{}) : small(CuSmallSum<false>{});
}
template <int N>
int launch_copy(const Plan& plan, hipStream_t stream) {
    using Large = std::conditional_t<(N > 2), CuLargeCopies<N>, CuLargeCopy>;
    if constexpr (N >= kCuVastCopies)
        if (plan.cu_far) return launch_as<&cu_ring_copy_kernel<N, CuVastCopies, true>, N, true>(plan, stream);
    if (plan.cu_large) return launch_as<&cu_ring_copy_kernel<N, Large, true>, N, true>(plan, stream);
    const auto small = [&](auto form) {
        using Small = decltype(form);
        if (plan.cu_args.split) return launch_as<&cu_ring_copy_kernel<N, Small, true>, N, true>(plan, stream);
        return launch_as<&cu_ring_copy_kernel<N, Small, false>, N, false>(plan, stream);
    };
    if constexpr (N > 2) return small(CuSmall<true>{});
    else return plan.cu_through ? small(CuSmall<true>{}) : small(CuSmall<false>{});
}

template <int N>
int launch_ranks(const Plan& plan, int dtype, hipStream_t stream) {
    const bool everywhere = plan.cu_args.op == OP_ALLREDUCE;
    switch (dtype) {
        case MINT_F16: return everywhere ? launch_sum<DT_F16, N, true>(plan, stream)
                                         : launch_sum<DT_F16, N, false>(plan, stream);
        case MINT_BF16: return everywhere ? launch_sum<DT_BF16, N, true>(plan, stream)
                                          : launch_sum<DT_BF16, N, false>(plan, stream);
        case MINT_F32: return everywhere ? launch_sum<DT_F32, N, true>(plan, stream)
                                         : launch_sum<DT_F32, N, false>(plan, stream);
        default: return launch_copy<N>(plan, stream);
    }
}

int launch_alltoall(const Plan& plan, hipStream_t stream) {
    const CuRingArgs& a = plan.cu_args;
    const CuShape& s = a.shape;
    CuPairs<uint64_t> far = {};
    CuPairs<uint32_t> near = {};
    uint64_t lowest = ~0ull, rest = 0;            // rest: what the short form cannot say
    for (uint32_t i = 0; i < a.len; ++i) {
        far.rank[i] = a.input[i];
        far.rank[kMaxRanks + i] = a.output[i];
        lowest = std::min({lowest, a.input[i], a.output[i]});
    }
    for (uint32_t i = 0; i < 2 * kMaxRanks; ++i) {
        const uint64_t off = far.rank[i] ? far.rank[i] - lowest : 0;
        near.rank[i] = (uint32_t)(off >> kCuNearShift);
        rest |= off ^ (uint64_t)near.rank[i] << kCuNearShift;
    }
    const dim3 grid = grid_of(plan, a.len, a.len);
    const unsigned threads = (unsigned)plan.threads;
    const u32x2 counts = {s.tiles, s.part};
    const u64x4 numbers = {s.row_bytes, s.row_stride, lowest, reinterpret_cast<uint64_t>(a.status)};
    if (plan.cu_large)
        return Launch<&cu_alltoall_kernel<CuLargeCopy, uint64_t>>::go(grid, threads, 0, stream, numbers, counts, far);
    const auto small = [&](auto form) {
        using Small = decltype(form);
        if (rest) return Launch<&cu_alltoall_kernel<Small, uint64_t>>::go(grid, threads, 0, stream, numbers, counts, far);
        return Launch<&cu_alltoall_kernel<Small, uint32_t>>::go(grid, threads, 0, stream, numbers, counts, near);
    };
    return plan.cu_through ? small(CuSmall<true>{}) : small(CuSmall<false>{});
}

}  // namespace

int launch_cu_ring(const Plan& plan, int dtype, hipStream_t stream) {
    if (plan.cu_args.op == OP_ALLTOALL) return launch_alltoall(plan, stream);
    switch (plan.cu_args.len) {
        case 2: return launch_ranks<2>(plan, dtype, stream);
        case 3: return launch_ranks<3>(plan, dtype, stream);
        case 4: return launch_ranks<4>(plan, dtype, stream);
        case 5: return launch_ranks<5>(plan, dtype, stream);
        case 6: return launch_ranks<6>(plan, dtype, stream);
        case 7: return launch_ranks<7>(plan, dtype, stream);
        case 8: return launch_ranks<8>(plan, dtype, stream);
        default: return MINT_ERR_ARG;
    }
}

}  // namespace mint
