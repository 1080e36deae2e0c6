// The requests for attn_bias of a wavefront of hstu_bwd_kv_fused_kernel, step after step: the plane of the query head, whose first byte
// and size make the descriptor, and a byte offset per lane.  No device code: a host test replays them against the tensor's bounds.
#pragma once
#include <stdint.h>

#ifdef __HIP__
#include <hip/hip_runtime.h>
#define HSTU_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define HSTU_HOST_DEVICE inline
#endif

namespace hstu {

constexpr uint32_t kPastPlane = 0x80000000u;  // a byte offset no plane contains (the host takes planes below 2 GiB), nor with a row's offset added

struct BiasRequests {
    uint64_t plane;    // address of the query head's plane
    uint32_t pitch;    // bytes of a row
    uint32_t size;     // bytes of a plane
    uint32_t lane;     // the lane's offset in the rows of query sub-tile 0
    int x, first, skip_from, skip_to, end;  // the next query sub-tile; behind skip_from - 1 comes skip_to, behind end - 1 the next head's first
    int left;          // steps that still need one

    // Lane (ln, lh) has row ln of a sub-tile, the 16 bytes of keys cw0 + 8 lh .. + 7 and the 16 bytes 32 further on.
    HSTU_HOST_DEVICE void set_lane(int max_k, int cw0, int ln, int lh)
    {
        lane = cw0 + 8 * lh < max_k ? static_cast<uint32_t>(ln) * pitch + static_cast<uint32_t>(cw0 + 8 * lh) * 2u : kPastPlane;
    }
    // The descriptor's size.  The request behind the last step is sent like the others, so that a step waits by one count: its
    // descriptor is empty.  (An offset added to kPastPlane would not do: a second kPastPlane wraps to 0.)
    HSTU_HOST_DEVICE uint32_t bytes() const { return left > 0 ? size : 0u; }
    HSTU_HOST_DEVICE uint32_t offset() const { return lane + static_cast<uint32_t>(x * 32) * pitch; }
    HSTU_HOST_DEVICE void advance()
    {
        --left;
        if (++x == skip_from) {
            x = skip_to;
        }
        if (x >= end) {
            x = first;
            plane += left > 0 ? size : 0u;
        }
    }
};

}  // namespace hstu
