// Device helpers of the solves that run as one launch (resident.hip, resident_ic0.hip).
#pragma once

#include "device.hpp"
#include "sync.hpp"

namespace pfem {

// Compute units for the workgroups of such a solve, held from its launch to its end: the solves of several threads
// (contexts) of one process run side by side only while all their workgroups fit the device together, since they
// could otherwise share it so that none is complete, and all would wait out their limits. One unit a workgroup
// is enough however they are placed; workgroups are dealt to the XCDs in turn, so a solve takes as many of each of
// the eight as it can have on one. A solve of more workgroups than units (several to a unit) has the device
// to itself. Solves are admitted in the order they come. 8 threads with 5 (39) workgroups each, ten solves each:
// 66 (287) ms against 153 (618) one after the other.
class ResidentSeats {
public:
    ResidentSeats(int device, int blocks, int cus);
    ~ResidentSeats();
    ResidentSeats(const ResidentSeats&) = delete;
    ResidentSeats& operator=(const ResidentSeats&) = delete;

private:
    int device_, taken_;
};

constexpr int kResPause = 64;   // solves that take the other path after a wait has failed

// Values the first poll does not find are polled until they are published, the limit is reached or another
// workgroup has given up.
template <typename T>
__device__ __forceinline__ T res_await(typename Sentinel<T>::U* q, typename Sentinel<T>::U v, int* err, long limit,
                                       int* fail)
{
    constexpr typename Sentinel<T>::U sent = Sentinel<T>::bits;
    for (long spins = 0; v == sent; ++spins) {
        if (spins >= limit || ((spins == 63 || (spins & 1023) == 1023) &&
                               __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
            *fail = 1;
            __hip_atomic_fetch_max(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // (a 2 stays)
            break;
        }
        // workgroups of a batch's next system may wait for its last ones to start: they must not crowd the
        // fabric that the running systems exchange through
        if (spins >= 16) __builtin_amdgcn_s_sleep(16);
        v = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return __builtin_bit_cast(T, v);
}

// A value that is the same in every lane, kept in scalar registers
__device__ __forceinline__ double uniform(double t)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, t);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// ((v0 + v1) + v2) + v3 of lanes i .. i + 3 (within 16), in lane i: the order block_sum adds its waves in
__device__ __forceinline__ double sum4(double v)
{
    return ((v + lane_down<1>(v)) + lane_down<2>(v)) + lane_down<3>(v);
}

}  // namespace pfem
