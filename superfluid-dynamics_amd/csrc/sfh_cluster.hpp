// sfh_cluster.hpp -- several workgroups on one surface of the batched stage kernel.
//
// An ensemble of fewer surfaces than CUs leaves CUs idle, and its stage takes as long as its largest surface.  The
// host then launches up to kMaxParts workgroups for a large surface.  They repeat the node-local work (derivatives,
// Gram-Schmidt) and share the pair sweeps and the products of the stored matrix, which are split into a fixed number
// of parts: after a sweep each part's node sums go to an exchange buffer, the workgroups meet, and all add the parts
// in the same order.  So every workgroup holds the same values, takes the same branches, and a result does not
// depend on how many workgroups there are for the parts.
//
// Joining.  Nothing promises that the workgroups of a surface run at the same time.  Each takes a ticket; the first
// one waits a short while for the others and then closes the list.  Whoever comes later leaves at once, and the
// members share out its parts.  After that only members wait for each other, all of which are running: no wait
// depends on a workgroup that has not started.  (Waits also end after 2 s, which the host reports as an error.)  The
// last workgroup to leave, member or not, clears the words for the next launch.
//
// Exchange.  The sums are stored and loaded with agent scope, so they go past the XCDs' separate L2 caches; a store
// has arrived when its wave's vmcnt is 0, after which the workgroup counts itself in.  A release fence at agent
// scope would write back the L2's dirty matrix lines, which no other workgroup reads.  Two buffers alternate: a
// workgroup can only write one again after a meeting that all reach after reading it.
#pragma once
#include "sfh_kernels.hpp"

namespace sfh {

struct Cluster {
    int parts, launched;   // of the surface: parts of its work, workgroups
    int rank, members;
    int met;           // meetings so far
    bool gave_up;      // thread 0: a wait ended at its limit, later ones don't wait
    double* xb;        // two buffers of parts * kMaxSums * n sums
    int* words;        // ticket (and closed flag), members, count of the meetings, leavers
    int* failed;       // set when a wait gave up

    static constexpr int kClosed = 1 << 30;
    static constexpr int kMaxSums = 4;   // sums per node and part of one exchange

    __device__ static int load(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
    __device__ static int add(int* p, int v) {
        return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ static unsigned long long ticks() { return __builtin_amdgcn_s_memrealtime(); }   // 100 MHz

    // One thread: *p >= least, for at most the given time.
    __device__ static bool wait(const int* p, int least, unsigned long long limit) {
        const unsigned long long t0 = ticks();
        while ((load(p) & ~kClosed) < least) {
            if (ticks() - t0 > limit) return false;
            __builtin_amdgcn_s_sleep(1);
        }
        return true;
    }
    static constexpr unsigned long long kJoin = 2000, kGiveUp = 200000000;   // 20 us, 2 s

    __device__ void give_up(bool yes) {
        gave_up = yes;
        if (yes) *failed = 1;
    }

    // Thread 0, with the workgroup's ticket: rank and members (0: too late, leave).
    __device__ void join(int ticket) {
        rank = ticket & ~kClosed;
        if (ticket & kClosed) {
            members = 0;
        } else if (rank == 0) {
            wait(words, parts, kJoin);
            members = __hip_atomic_fetch_or(words, kClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(words + 1, members, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            give_up(!wait(words + 1, 1, kGiveUp));
            members = load(words + 1);
        }
    }
    // Thread 0, when this workgroup needs the words no more.
    __device__ void leave() {
        if (add(words + 3, 1) != launched - 1) return;
        for (int i = 0; i < 4; ++i) __hip_atomic_store(words + i, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    __device__ double* buffer(int n) const { return xb + (size_t)(met & 1) * parts * kMaxSums * n; }
    __device__ void put(int n, int slot, double v) {
        __hip_atomic_store(buffer(n) + (size_t)slot * n + threadIdx.x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // After the puts of this workgroup: all members' have arrived.
    __device__ void meet() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) {
            add(words + 2, 1);
            if (!gave_up) give_up(!wait(words + 2, members * (met + 1), kGiveUp));
        }
        __syncthreads();
    }
    // Meets, then out[a] = sum over the parts of slots p NA + a, on threads < n (0 on the others).
    template <int NA>
    __device__ void exchange(int n, double (&out)[NA]) {
        meet();
        const double* b = buffer(n) + min((int)threadIdx.x, n - 1);
        double v[kMaxParts][NA];
#pragma unroll
        for (int p = 0; p < kMaxParts; ++p)
#pragma unroll
            for (int a = 0; a < NA; ++a)   // clamped: every load in flight together
                v[p][a] = __hip_atomic_load(b + (size_t)(min(p, parts - 1) * NA + a) * n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            out[a] = 0.0;
#pragma unroll
            for (int p = 0; p < kMaxParts; ++p) out[a] += p < parts ? v[p][a] : 0.0;
            if ((int)threadIdx.x >= n) out[a] = 0.0;
        }
        ++met;
    }
    // Sum of one value per workgroup (the same in all its threads), in the members' order.
    __device__ double sum_members(int n, double v) {
        if (threadIdx.x == 0) put(n, rank, v);
        meet();
        double s = 0.0;
        for (int r = 0; r < members; ++r)
            s += __hip_atomic_load(buffer(n) + (size_t)r * n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ++met;
        return s;
    }
};

}  // namespace sfh
