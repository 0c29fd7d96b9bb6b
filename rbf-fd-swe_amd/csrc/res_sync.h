// Cross-workgroup exchange of the resident whole-step kernels: neighbour
// waits, stage counts and agent-coherent state accesses.
//
// The L2 caches of the 8 XCDs are not coherent with each other, so every
// state access another workgroup depends on is agent-coherent (direct-to-LDS
// loads and buffer stores with the sc1 cache policy; the published states
// are small and live in the last-level cache), and the stage counts are
// agent-scope atomics written after the state stores have completed.  Every
// wait is bounded (spin_limit polls): a workgroup that exceeds it raises the
// abort flag, which every waiting workgroup sees, and all of them leave the
// kernel; the host reports the launch as failed.
#pragma once

#include "swe_ctx.h"

namespace swe {

// Synchronisation state (unsigned words), zeroed before the first launch of
// a context and when the counts near 2^31: word 0 is the abort flag, then
// one 128-byte line per tile holding the number of stages the tile has
// completed, counted on across launches.  Instead of a grid-wide barrier a
// tile waits, before each stage, for the tiles it exchanges rows with (the
// owners of the rows it reads and the tiles that read its rows): they have
// then finished the previous stage, so the rows it reads are final and
// nobody still reads the buffer it is about to overwrite.  Neighbouring
// tiles are at most one stage apart and no wait depends on a later stage.
constexpr int kResLine = 32;

struct DevResSync {
    unsigned *sync;         // [1 + ntiles][kResLine]
    unsigned *host_abort;   // pinned host word, set on a time-out
    const int *nbrs;        // [ntiles][kResMaxNbrs] tiles to wait for, -1 padded
    unsigned stage0;        // stages completed before this launch
    unsigned spin_limit;
};

__device__ __forceinline__ unsigned ld_agent(const unsigned *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void st_agent(unsigned *p, unsigned v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wave 0 polls the neighbour tiles' stage counts (one per lane) until every
// one has reached `need`; false once any wait in the grid was aborted.  The
// lanes without a neighbour read the abort word in the same load (a second
// load per poll cost 0.05 us a stage).
__device__ __forceinline__ bool res_wait(const DevResSync &r, int tile, unsigned need)
{
    __shared__ int ok;
    if (threadIdx.x < 64) {
        const int u = r.nbrs[tile * kResMaxNbrs + (int)threadIdx.x];
        const unsigned *f = u >= 0 ? r.sync + (long)(1 + u) * kResLine : r.sync;
        const bool watched = __any(u < 0);
        int good = 1;
        unsigned polls = 0;
        for (;;) {
            const unsigned v = ld_agent(f);
            if (!__any(u >= 0 && v < need))
                break;
            if (++polls > r.spin_limit || __any(u < 0 && v != 0)
                || (!watched && ld_agent(r.sync))) {
                if (threadIdx.x == 0) {
                    st_agent(r.sync, 1u);
                    __hip_atomic_store(r.host_abort, 1u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_SYSTEM);
                }
                good = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        if (threadIdx.x == 0)
            ok = good;
    }
    __syncthreads();
    return ok != 0;
}

// Every wave's state stores are complete, then the tile's count moves on.
__device__ __forceinline__ void res_publish(const DevResSync &r, int tile, unsigned done)
{
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0)
        st_agent(r.sync + (long)(1 + tile) * kResLine, done);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t state_rsrc(const void *p, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, bytes, 0x00020000);
}

constexpr int kSc1 = 16;   // cache policy: agent-coherent access

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes per lane from global memory straight into LDS, agent-coherent
// (global_load_lds_dwordx4 ... sc1): lane l's bytes land at lds + 16 l, lds
// being wave-uniform; the wave's vmcnt counts the load until they are there.
__device__ __forceinline__ void dma16_sc1(const void *src, void *lds)
{
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void *)lds, 16, 0,
                                     kSc1);
}

}  // namespace swe
