// The LL128 codec, wave64 layout (protocol.hpp): a message from raw bytes and back.
//
// Bound by memory from some MiB on.  A wavefront moves one block of the message and ends (the
// loop is for messages beyond 2^31 threads), so that what is in flight is one
// window that moves through memory; the lines go through the L2 into the last-level
// cache for whoever unpacks them, the raw bytes that unpack leaves past it.
// pack + unpack, resident wavefronts that stride / a wavefront per block and plain
// stores / this: 16 MiB 14.1 / 13.7 / 13.0 us, 32 MiB 25.6 / 22.8 / 22.2, 48 MiB 36.7 /
// 34.7 / 32.4, 64 MiB 47.0 / 45.4 / 42.4 (blocks of 256 threads 1 - 3 % slower, of 64 within
// 1 %); which thread blocks an XCD takes: launch_wave64.
//
// With a KiB to a wavefront, what stands before its load counts.  All numbers in registers when it
// starts, one test for the ragged last block, lanes told apart by selects (13 scalar and 20 vector
// instructions to the load) over numbers read from memory and two paths at each of the three (45, six
// branches): pack + unpack, three sets of buffers in turn / 750 MiB between two uses, us: 8 MiB 8.2 -> 7.2 /
// 9.6 -> 8.4, 16 MiB 12.4 -> 11.6 / 14.5 -> 13.0, 32 MiB 21.2 -> 20.6 / 24.7 -> 23.4, 64 MiB 43.0 -> 41.3 (6.7 TB/s, a
// copy's rate) / 43.9 -> 42.2.  Below 5 MiB the host's two launches are what it takes.
#include "ring_launch.hpp"

namespace mint {
namespace {

constexpr uint32_t kCodecThreads = 128;

// A launch has at most 2^31 threads; a wavefront that has moved its block goes on with the one that many
// wavefronts further, if there is any.
constexpr uint32_t kCodecMostBlocks = (1u << 31) / kCodecThreads, kCodecMostWaves = kCodecMostBlocks * (kCodecThreads / 64u);

// All of a launch's numbers fit into the 14 words that arrive in registers, in two arguments (each
// costs a launch 10 ns): `a`: where from, where to, raw bytes, blocks of the message, of them
// whole ones if kCodecRagged is not set | part << 32; `b`: flag base, flag stride (a sector's tag is the low
// half of its line's flag), the counter of bad flags.
//
// The blocks of the message that a wavefront moves: `part` > 0, an XCD `part` thread blocks' worth of
// consecutive ones (see CuPlace: the hardware deals thread blocks to the eight XCDs in turn).  The last
// block of the message, if the raw bytes end inside it, is moved byte by byte, away from the
// others' path.
constexpr uint32_t kCodecRagged = 1u << 31;
struct CodecWaves {
    uint32_t first, blocks, whole;
    __device__ __forceinline__ CodecWaves(uint64_t counts) {
        uint32_t part = (uint32_t)(counts >> 32);
        const uint32_t x = blockIdx.x;
        asm volatile("" : "+s"(part));             // (or the compiler compares and branches on all 64 bits)
        const uint32_t at = part ? (x & 7u) * part + (x >> 3) : x;
        first = __builtin_amdgcn_readfirstlane(at * (kCodecThreads / 64u) + (uint32_t)wave_in_block());
        blocks = (uint32_t)counts & ~kCodecRagged;
        whole = blocks - ((uint32_t)counts >> 31);
    }
    template <typename WHOLE, typename RAGGED>
    __device__ __forceinline__ void each(const WHOLE& whole_block, const RAGGED& ragged_block) const {
        uint32_t g = first;
#pragma unroll 1
        for (; g < whole; g += kCodecMostWaves) whole_block(g);
        if (__builtin_expect(g == whole && g < blocks, 0)) ragged_block(g);
    }
};
// LaneMap of this lane, by selects of two values: what the compiler makes of LaneMap's own
// constructor are two paths with half of the lanes each.
__device__ __forceinline__ LaneMap codec_lanes() {
    LaneMap m;
    uint32_t vector = (m.lane - m.sector) * 16u, tagged = kFlagLaneRaw + 12u * m.sector;
    asm volatile("" : "+v"(vector), "+v"(tagged));
    m.raw_off = m.flag_lane ? tagged : vector;
    return m;
}
// the tag of both sectors of this lane's line (two sectors to a line)
__device__ __forceinline__ uint32_t codec_tag(uint32_t g, const LaneMap& m, u32x4 b) {
    return b.x + (g * 8u + (m.sector >> 1)) * b.y;
}

__global__ void __launch_bounds__(kCodecThreads) pack_wave64_kernel(u64x4 a, u32x4 b) {
    const uint8_t* const raw = reinterpret_cast<const uint8_t*>(a.x);
    uint8_t* const msg = reinterpret_cast<uint8_t*>(a.y);
    const CodecWaves w(a.w);
    const LaneMap m = codec_lanes();
    const uint32_t lane_off = m.raw_off - (m.flag_lane ? 4u : 0u);
    const auto store = [&](uint32_t g, u32x4 v) MINT_INLINE_LAMBDA {
        st128_through<false>(msg + (uint64_t)g * kBlockMsg, m.lane * 16u, v);
    };
    w.each(
        [&](uint32_t g) MINT_INLINE_LAMBDA {
            const u32x4 v = *(MINT_GLOBAL const u32x4_a1*)(as_global(raw + (uint64_t)g * kBlockRawLL) + lane_off);
            uint32_t tag = codec_tag(g, m, b);
            asm volatile("" : "+v"(tag));
            store(g, u32x4{m.flag_lane ? v.y : v.x, m.flag_lane ? v.z : v.y, m.flag_lane ? v.w : v.z, m.flag_lane ? tag : v.w});
        },
        [&](uint32_t g) MINT_INLINE_LAMBDA {
            u32x4 v = load_guarded(raw, (uint64_t)g * kBlockRawLL + m.raw_off, m.raw_len, a.z);
            if (m.flag_lane) v.w = codec_tag(g, m, b);
            store(g, v);
        });
}
__global__ void __launch_bounds__(kCodecThreads) unpack_wave64_kernel(u64x4 a, u32x4 b) {
    const uint8_t* const msg = reinterpret_cast<const uint8_t*>(a.x);
    uint8_t* const raw = reinterpret_cast<uint8_t*>(a.y);
    unsigned long long* const bad_flags = reinterpret_cast<unsigned long long*>((uint64_t)b.w << 32 | b.z);
    const CodecWaves w(a.w);
    const LaneMap m = codec_lanes();
    uint32_t bad = 0;
    const auto load = [&](uint32_t g) MINT_INLINE_LAMBDA {
        const u32x4 v = *(MINT_GLOBAL const u32x4*)(as_global(msg + (uint64_t)g * kBlockMsg) + m.lane * 16u);
        if (bad_flags) {
            // a line is bad if either of its two sector tags is (flag lanes 3 and
            // 7 of every 8); count it once
            uint64_t wrong = __ballot(m.flag_lane && v.w != codec_tag(g, m, b));
            wrong |= wrong << 4;
            bad += (uint32_t)__popcll(wrong & 0x8080808080808080ull);
        }
        return v;
    };
    w.each(
        [&](uint32_t g) MINT_INLINE_LAMBDA {
            const u32x4 v = load(g);
            uint8_t* const to = raw + (uint64_t)g * kBlockRawLL;
            if (m.flag_lane) st96_through<true>(to, m.raw_off, u32x3{v.x, v.y, v.z});
            else st128_through<true>(to, m.raw_off, v);
        },
        [&](uint32_t g) MINT_INLINE_LAMBDA { store_guarded(raw, (uint64_t)g * kBlockRawLL + m.raw_off, m.raw_len, a.z, load(g)); });
    if (bad && lane_id() == 0) atomicAdd(bad_flags, (unsigned long long)bad);
}

// One wavefront per block of the message, but no more threads than a launch may have.  An
// XCD takes consecutive thread blocks between the sizes where
// that is measured to be faster.  pack + unpack, dealt one by one (and with eight launch arguments) / so, us,
// the same buffers again, three sets in turn, 750 MiB between two uses: 4 MiB 6.4 / 6.1, 6.4 / 6.2, 7.0 / 6.7; 8 MiB 7.4 / 7.2, 8.4 / 8.2, 9.6 /
// 9.6; 16 MiB 12.2 / 11.0, 12.9 / 12.4, 14.7 / 14.6; 32 MiB 22.1 / 21.2, 22.0 / 21.1, 24.5 / 24.8; 48 MiB 31.1 /
// 30.3, 32.6 / 32.2, 34.0 / 33.4; 59 MiB 37.4 / 36.5, 39.6 / 38.5, 40.5 / 39.8; at 64 MiB, three sets, 41.2 /
// 42.1.
template <auto KERNEL>
int launch_wave64(const void* from, void* to, uint64_t nbytes, uint64_t lines, uint64_t flag_base, uint64_t flag_stride, void* bad,
                  hipStream_t stream) {
    const uint64_t wanted = (lines * 8 + kCodecThreads - 1) / kCodecThreads;
    uint32_t blocks = wanted > kCodecMostBlocks ? kCodecMostBlocks : (uint32_t)wanted, part = 0;
    if (nbytes >= (4ull << 20) && nbytes <= (60ull << 20)) {
        part = (blocks + kXcds - 1) / kXcds;
        blocks = part * kXcds;
    }
    const uint64_t ragged = nbytes % kBlockRawLL ? kCodecRagged : 0u, counter = reinterpret_cast<uint64_t>(bad);
    const u64x4 a = {reinterpret_cast<uint64_t>(from), reinterpret_cast<uint64_t>(to), nbytes, (uint64_t)part << 32 | ragged | lines / 8};
    const u32x4 b = {(uint32_t)flag_base, (uint32_t)flag_stride, (uint32_t)counter, (uint32_t)(counter >> 32)};
    return Launch<KERNEL>::go(blocks, kCodecThreads, 0, stream, a, b);
}

}  // namespace

int launch_pack_wave64(const void* raw, void* msg, uint64_t nbytes, uint64_t lines, uint64_t flag_base, uint64_t flag_stride,
                       hipStream_t stream) {
    return launch_wave64<&pack_wave64_kernel>(raw, msg, nbytes, lines, flag_base, flag_stride, nullptr, stream);
}
int launch_unpack_wave64(const void* msg, void* raw, uint64_t nbytes, uint64_t lines, uint64_t flag_base, uint64_t flag_stride,
                         void* bad_flags, hipStream_t stream) {
    return launch_wave64<&unpack_wave64_kernel>(msg, raw, nbytes, lines, flag_base, flag_stride, bad_flags, stream);
}

}  // namespace mint
