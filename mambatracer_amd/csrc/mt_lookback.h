// Decoupled look-back over tiles, shared by the scans and compactions
// (mt_scan.hip, described there) and the BVH builder's fused flag scan
// (mt_bvh.hip).
#pragma once
#include "mt_devmath.h"
#include "mt_internal.h"

namespace {

constexpr uint32_t FLAG_AGG = 1u, FLAG_INC = 2u;
constexpr uint32_t SPIN_LIMIT = 1u << 26;

struct ScanWork {
    uint32_t* ticket; // [0] ticket, [1] error flag (spin limit hit), [2] epoch of the current call
    uint64_t* status; // [ntiles]
};

__device__ __forceinline__ uint64_t pack_status(uint32_t epoch, uint32_t flag, uint32_t v)
{
    return ((uint64_t)(epoch & 0x3FFFFFFFu) << 34) | ((uint64_t)flag << 32) | (uint64_t)v;
}

__device__ __forceinline__ int lane_id() { return __lane_id(); }

// Decoupled look-back by wave 0 of the tile.  Returns the exclusive prefix of
// `tile` (all lanes of wave 0 agree); publishes the tile's inclusive prefix.
__device__ uint32_t look_back(ScanWork W, int tile, uint32_t aggregate, uint32_t epoch)
{
    const int lane = lane_id();
    uint64_t* st = W.status;
    if (tile == 0) {
        if (lane == 0)
            __hip_atomic_store(&st[0], pack_status(epoch, FLAG_INC, aggregate), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        return 0u;
    }
    if (lane == 0)
        __hip_atomic_store(&st[tile], pack_status(epoch, FLAG_AGG, aggregate), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    uint32_t prefix = 0;
    int window_end = tile - 1; // predecessor examined by lane 0
    const uint32_t ep = epoch & 0x3FFFFFFFu;
    uint32_t spins = 0;
    for (;;) {
        int idx = window_end - lane;
        uint64_t w;
        uint32_t flag, val;
        for (;;) {
            if (idx >= 0) {
                w = __hip_atomic_load(&st[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                bool cur = (uint32_t)(w >> 34) == ep;
                flag = cur ? (uint32_t)(w >> 32) & 3u : 0u;
                val = (uint32_t)w;
            } else { // before tile 0: an inclusive zero
                flag = FLAG_INC;
                val = 0;
            }
            if (__all(flag != 0)) break;
            if (++spins > SPIN_LIMIT) {
                if (lane == 0) atomicOr(&W.ticket[1], 1u);
                return prefix; // results invalid; the host reports the error flag
            }
            __builtin_amdgcn_s_sleep(1);
        }
        uint64_t inc = __ballot(flag == FLAG_INC);
        // lanes up to and including the nearest inclusive predecessor contribute
        int first_inc = inc ? __builtin_ctzll(inc) : 64;
        uint32_t contrib = lane <= first_inc ? val : 0u;
        for (int o = 32; o > 0; o >>= 1) contrib += __shfl_xor(contrib, o);
        prefix += contrib;
        if (inc) break;
        window_end -= 64;
    }
    if (lane == 0)
        __hip_atomic_store(&st[tile], pack_status(epoch, FLAG_INC, prefix + aggregate),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return prefix;
}

// The context's look-back workspace for ntiles tiles (grown as needed).
inline int32_t scan_workspace_tiles(mt_context* ctx, int64_t ntiles, ScanWork& W)
{
    size_t bytes = 256 + sizeof(uint64_t) * (size_t)(ntiles > 0 ? ntiles : 1);
    void* p = nullptr;
    int32_t rc = mt_ctx_scratch(ctx, bytes, &p);
    if (rc) return rc;
    W.ticket = reinterpret_cast<uint32_t*>(p);
    W.status = reinterpret_cast<uint64_t*>(reinterpret_cast<char*>(p) + 256);
    return MT_OK;
}

} // namespace
