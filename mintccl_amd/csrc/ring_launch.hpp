// Host side of the ring kernels: the launch plan and one launcher per element
// type.  Each launcher lives in a translation unit of its own (ring_family.hip
// compiled with MINT_FAMILY_DT = 0..3), which lets the build compile the four
// kernel families in parallel.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

#include "../../include/mintccl.h"
#include "cu_ring.hpp"
#include "ring.hpp"

namespace mint {

struct Plan {
    RingArgs args;
    int blocks, threads, unroll;
    int blocks_plain;         // the grid without CUs set apart for origins (args.origin_cus)
    size_t staging_need;      // bytes of staging per rank: slots + credit words
    bool empty;
    bool lds;                 // own rows through LDS: `threads` counts the wave-channels'
                              // threads only, the launch adds the fetcher wavefront
    bool cu;                  // rings inside compute units: `cu_args` instead of `args`
    CuRingArgs cu_args;
    CuChoice cu_choice;       // ... and the form of their kernels
    int cu_lds;               // bytes of LDS per block, to bound how many a compute unit holds
};

inline int launch_status() { return hipGetLastError() == hipSuccess ? MINT_OK : MINT_ERR_HIP; }

constexpr int kDevices = 16;      // per-device facts are kept for the first so many
inline int device_cus() {
    static std::atomic<int> known[kDevices];
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (dev < kDevices && (cus = known[dev].load(std::memory_order_relaxed)) != 0) return cus;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    if (dev < kDevices) known[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// The calling thread's device.  Where there is only one there is nothing to ask
// (hipGetDevice takes 0.05 us, a launch 2.6).
inline bool this_device(int* dev) {
    static const bool only = [] {
        int n = 0;
        return hipGetDeviceCount(&n) == hipSuccess && n == 1;
    }();
    *dev = 0;
    return only || hipGetDevice(dev) == hipSuccess;
}

// Launches KERNEL.  A launch costs the host 2.7 us and is most of what a small
// collective takes (4.0), so the symbol is looked up once per device and not on
// every launch (<<<>>>: 2.8).
template <auto KERNEL>
struct Launch;
template <typename... P, void (*KERNEL)(P...)>
struct Launch<KERNEL> {
    static int go(dim3 grid, unsigned threads, unsigned lds_bytes, hipStream_t stream, const P&... args) {
        static std::atomic<hipFunction_t> known[kDevices];
        int dev;
        if (!this_device(&dev)) return MINT_ERR_HIP;
        hipFunction_t f = dev < kDevices ? known[dev].load(std::memory_order_acquire) : nullptr;
        if (!f) {
            if (hipGetFuncBySymbol(&f, reinterpret_cast<const void*>(KERNEL)) != hipSuccess) return MINT_ERR_HIP;
            if (dev < kDevices) known[dev].store(f, std::memory_order_release);
        }
        void* list[] = {const_cast<void*>(static_cast<const void*>(&args))...};
        const hipError_t e = hipModuleLaunchKernel(f, grid.x, grid.y, grid.z, threads, 1, 1, lds_bytes, stream,
                                                   list, nullptr);
        return e == hipSuccess ? MINT_OK : MINT_ERR_HIP;
    }
};

// protocol: MINT_PROTO_*; cache_policy: 0 agent, 1 system, 2 XCD-local
int launch_ring_family_f16(const Plan& plan, int protocol, int cache_policy, hipStream_t stream);
int launch_ring_family_bf16(const Plan& plan, int protocol, int cache_policy, hipStream_t stream);
int launch_ring_family_f32(const Plan& plan, int protocol, int cache_policy, hipStream_t stream);
int launch_ring_family_bytes(const Plan& plan, int protocol, int cache_policy, hipStream_t stream);
int launch_cu_ring(const Plan& plan, int dtype, hipStream_t stream);
// the codec, wave64 layout (codec.hip): `lines` of the message, whole blocks of eight
int launch_pack_wave64(const void* raw, void* msg, uint64_t nbytes, uint64_t lines, uint64_t flag_base, uint64_t flag_stride,
                       hipStream_t stream);
int launch_unpack_wave64(const void* msg, void* raw, uint64_t nbytes, uint64_t lines, uint64_t flag_base, uint64_t flag_stride,
                         void* bad_flags, hipStream_t stream);

}  // namespace mint
