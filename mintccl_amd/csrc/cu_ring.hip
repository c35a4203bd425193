// The kernels of rings inside compute units (cu_ring.hpp) and their launcher.
#include "ring_launch.hpp"

namespace mint {
namespace {

// A block is a whole channel and nobody waits for another block, so a grid of
// any size will do.
template <int DT, int U, int NS, int D>
int launch_as(const Plan& plan, hipStream_t stream) {
    const size_t lds_bytes = kCuWordBytes + (size_t)plan.cu_args.hops * NS * U * kBlockRawSimple;
    hipLaunchKernelGGL((cu_ring_kernel<DT, U, NS, D>), dim3((unsigned)plan.blocks),
                       dim3((unsigned)plan.threads), lds_bytes, stream, plan.cu_args);
    return launch_status();
}

}  // namespace

int launch_cu_ring(const Plan& plan, int dtype, hipStream_t stream) {
    switch (dtype) {
        case MINT_F16: return launch_as<DT_F16, 1, 4, 4>(plan, stream);
        case MINT_BF16: return launch_as<DT_BF16, 1, 4, 4>(plan, stream);
        case MINT_F32: return launch_as<DT_F32, 1, 4, 4>(plan, stream);
        default:
            if (plan.unroll == 1) return launch_as<DT_BYTES, 1, 4, 4>(plan, stream);
            return launch_as<DT_BYTES, 4, 2, 4>(plan, stream);
    }
}

}  // namespace mint
