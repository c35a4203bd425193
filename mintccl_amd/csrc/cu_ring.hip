// The kernels of rings inside compute units (cu_ring.hpp) and their launcher.
#include "ring_launch.hpp"

namespace mint {
namespace {

template <typename K>
int launch_as(K kernel, const Plan& plan, hipStream_t stream) {
    const CuRingArgs& a = plan.cu_args;
    const CuShape& s = a.shape;
    const uint32_t x = s.tiles + a.ends, y = a.op == OP_ALLTOALL ? a.len : a.pipes;
    const dim3 grid(plan.cu_large ? x : y, plan.cu_large ? y : x, a.op == OP_ALLTOALL ? a.len : 1u);
    hipLaunchKernelGGL(kernel, grid, dim3((unsigned)plan.threads), (unsigned)plan.cu_lds, stream, s.starts,
                       s.row_bytes, s.row_stride, s.short_bytes, s.full, s.tiles, a.tables);
    return launch_status();
}

template <int DT, int N>
int launch_sum(const Plan& plan, hipStream_t stream) {
    const bool everywhere = plan.cu_args.op == OP_ALLREDUCE;
    if (plan.cu_large)
        return everywhere ? launch_as(cu_ring_sum_kernel<DT, N, true, true>, plan, stream)
                          : launch_as(cu_ring_sum_kernel<DT, N, false, true>, plan, stream);
    return everywhere ? launch_as(cu_ring_sum_kernel<DT, N, true, false>, plan, stream)
                      : launch_as(cu_ring_sum_kernel<DT, N, false, false>, plan, stream);
}

template <int DT>
int launch_sum(const Plan& plan, hipStream_t stream) {
    switch (plan.cu_args.len) {
        case 2: return launch_sum<DT, 2>(plan, stream);
        case 3: return launch_sum<DT, 3>(plan, stream);
        case 4: return launch_sum<DT, 4>(plan, stream);
        case 5: return launch_sum<DT, 5>(plan, stream);
        case 6: return launch_sum<DT, 6>(plan, stream);
        case 7: return launch_sum<DT, 7>(plan, stream);
        case 8: return launch_sum<DT, 8>(plan, stream);
        default: return MINT_ERR_ARG;
    }
}

template <int COPIES, bool ALLTOALL = false>
int launch_copies(const Plan& plan, hipStream_t stream) {
    return plan.cu_large ? launch_as(cu_ring_copy_kernel<COPIES, ALLTOALL, true>, plan, stream)
                          : launch_as(cu_ring_copy_kernel<COPIES, ALLTOALL, false>, plan, stream);
}

int launch_copy(const Plan& plan, hipStream_t stream) {
    const CuRingArgs& a = plan.cu_args;
    if (a.op == OP_ALLTOALL) return launch_copies<1, true>(plan, stream);
    switch (a.op == OP_BROADCAST || a.op == OP_ALLGATHER ? a.len - 1 : 1) {
        case 1: return launch_copies<1>(plan, stream);
        case 2: return launch_copies<2>(plan, stream);
        case 3: return launch_copies<3>(plan, stream);
        case 4: return launch_copies<4>(plan, stream);
        case 5: return launch_copies<5>(plan, stream);
        case 6: return launch_copies<6>(plan, stream);
        case 7: return launch_copies<7>(plan, stream);
        default: return MINT_ERR_ARG;
    }
}

}  // namespace

int launch_cu_ring(const Plan& plan, int dtype, hipStream_t stream) {
    switch (dtype) {
        case MINT_F16: return launch_sum<DT_F16>(plan, stream);
        case MINT_BF16: return launch_sum<DT_BF16>(plan, stream);
        case MINT_F32: return launch_sum<DT_F32>(plan, stream);
        default: return launch_copy(plan, stream);
    }
}

}  // namespace mint
