// The kernels of rings inside compute units (cu_ring.hpp) and their launcher.
#include <algorithm>

#include "ring_launch.hpp"

namespace mint {
namespace {

// `rows`: pipelines, alltoall: destinations
template <typename FORM>
dim3 grid_of(const Plan& plan, uint32_t rows, uint32_t sources) {
    const CuRingArgs& a = plan.cu_args;
    const bool by_row = FORM::kLarge || a.shape.part;
    return dim3(by_row ? a.blocks : rows, by_row ? rows : a.blocks, sources);
}

template <typename FORM, auto KERNEL, int N, bool SPLIT>
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
    return Launch<KERNEL>::go(grid_of<FORM>(plan, a.pipes, 1), FORM::kThreads, (unsigned)plan.cu_lds, stream, numbers,
                              u32x2{s.tiles, s.part}, tables);
}

// use(what follows the rows and four words among the arguments of a launch by distances)
template <int N, typename USE>
int cu_near_more(const USE& use) {
    if constexpr (N <= 4) return use();
    else if constexpr (N <= 6) return use((uint64_t*)nullptr);
    else return use(u32x2{}, (uint64_t*)nullptr);
}
template <typename FORM, int N, auto KERNEL>
int launch_near(const Plan& plan, hipStream_t stream) {
    const CuRingArgs& a = plan.cu_args;
    const CuShape& s = a.shape;
    const dim3 grid = grid_of<FORM>(plan, a.pipes, 1);
    // (one pipeline: from its root on, so that the kernel has nothing to turn)
    const bool one = a.pipes == 1;
    uint32_t at[kMaxRanks] = {}, from = one ? s.starts : 0u;
    for (int i = 0; i < N; ++i) {
        at[i] = (uint32_t)((a.input[from] ? a.input[from] : a.output[from]) - a.lowest);
        from = from + 1 == N ? 0 : from + 1;
    }
    const bool cut = s.full < a.pipes;
    const u32x8 rows = {(uint32_t)a.lowest, (uint32_t)(a.lowest >> 32), (uint32_t)s.row_bytes,
                        (uint32_t)(cut ? s.short_bytes : s.row_stride), at[0], at[1], at[2], at[3]};
    const u32x2 counts = {(one ? 0u : s.starts) | s.full << 24 | (cut ? kCuNearCut : 0u), s.tiles | s.part << cu_near_part_bit(FORM::kLarge)};
    const auto go = [&](const auto&... words) {
        return Launch<KERNEL>::go(grid, FORM::kThreads, (unsigned)plan.cu_lds, stream, rows, words...);
    };
    const uint64_t status = reinterpret_cast<uint64_t>(a.status);
    if constexpr (N <= 4) return go(u32x4{counts.x, counts.y, (uint32_t)status, (uint32_t)(status >> 32)});
    else if constexpr (N <= 6) return go(u32x4{at[4], at[5], counts.x, counts.y}, a.status);
    else return go(u32x4{at[4], at[5], at[6], at[7]}, counts, a.status);
}

template <int DT, int N, bool EVERYWHERE>
int launch_sum(const Plan& plan, hipStream_t stream) {
    return cu_sum_form<N, EVERYWHERE>(plan.cu_choice, [&](auto form) {
        using Form = typename decltype(form)::type;
        if (plan.cu_args.near)
            return cu_near_more<N>([&](auto... more) {
                return launch_near<Form, N, &cu_near_sum_kernel<DT, N, EVERYWHERE, Form, decltype(more)...>>(plan, stream);
            });
        if constexpr (decltype(form)::in_place)
            if (!plan.cu_args.split)
                return launch_as<Form, &cu_ring_sum_kernel<DT, N, EVERYWHERE, Form, false>, N, false>(plan, stream);
        return launch_as<Form, &cu_ring_sum_kernel<DT, N, EVERYWHERE, Form, true>, N, true>(plan, stream);
    });
}
template <int N>
int launch_copy(const Plan& plan, hipStream_t stream) {
    return cu_copy_form<N>(plan.cu_choice, [&](auto form) {
        using Form = typename decltype(form)::type;
        if (plan.cu_args.near)
            return cu_near_more<N>([&](auto... more) {
                return launch_near<Form, N, &cu_near_copy_kernel<N, Form, decltype(more)...>>(plan, stream);
            });
        if constexpr (decltype(form)::in_place)
            if (!plan.cu_args.split) return launch_as<Form, &cu_ring_copy_kernel<N, Form, false>, N, false>(plan, stream);
        return launch_as<Form, &cu_ring_copy_kernel<N, Form, true>, N, true>(plan, stream);
    });
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
    const u32x2 counts = {s.tiles, s.part};
    const u64x4 numbers = {s.row_bytes, s.row_stride, lowest, reinterpret_cast<uint64_t>(a.status)};
    return cu_move_form(plan.cu_choice, [&](auto form) {
        using Form = typename decltype(form)::type;
        const dim3 grid = grid_of<Form>(plan, a.len, a.len);
        if constexpr (decltype(form)::in_place) {
            if (!rest && a.len <= kCuNearPairs && s.row_stride == s.row_bytes && s.tiles <= kCuNearTiles) {
                const uint32_t *from = near.rank, *to = near.rank + kMaxRanks;
                const u32x8 rows = {(uint32_t)lowest, (uint32_t)(lowest >> 32), (uint32_t)s.row_bytes,
                                    s.tiles | s.part << cu_near_part_bit(false), from[0], from[1], from[2], from[3]};
                return Launch<&cu_near_alltoall_kernel<Form>>::go(grid, Form::kThreads, 0, stream, rows, u32x4{to[0], to[1], to[2], to[3]},
                                                                  a.status);
            }
            if (!rest)
                return Launch<&cu_alltoall_kernel<Form, uint32_t>>::go(grid, Form::kThreads, 0, stream, numbers, counts, near);
        }
        return Launch<&cu_alltoall_kernel<Form, uint64_t>>::go(grid, Form::kThreads, 0, stream, numbers, counts, far);
    });
}

}  // namespace

int launch_cu_ring(const Plan& plan, int dtype, hipStream_t stream) {
    if (plan.cu_args.op == OP_ALLTOALL) return launch_alltoall(plan, stream);
    return cu_with_ranks((int)plan.cu_args.len, [&](auto ranks) {
        return launch_ranks<decltype(ranks)::value>(plan, dtype, stream);
    });
}

}  // namespace mint
