// ppl_dedisp_jobs.h -- what the dedispersion kernels share: the job table of
// a launch and small wait and barrier helpers.
#pragma once

#include "ppl_internal.h"

namespace ppl {

constexpr int kXcds = 8;

// One beam's part of a launch.  A launch covers several beams (jobs): job k
// owns workgroups [blockStart, blockStart + nDMTiles*nTTilesPad), a multiple
// of 8, so a job's own XCD-major tile order is kept.  The table travels in
// the kernel arguments; a workgroup finds its job with a uniform scan.
constexpr int kMaxDDJobs = PPL_DEDISP_MAX_JOBS;
struct DDJob {
    const void* in;
    void* out;
    const int32_t* delayT;
    int nChan, nsamp, tdms, tdmsPad, nOut;
    int rowUnits;   // LDS row length: elements (f32) or dwords per copy (f16, u8)
    int CB;         // channels per staged block
    int nDMTiles;
    int blockStart;
    int nTiles;     // tiles of the job (the window kernels' XCD split)
};
struct DDBatch {
    DDJob job[kMaxDDJobs];
    int n;
    float one;  // 1.0f, kept opaque to the compiler (f16 kernel)
};

__device__ __forceinline__ const DDJob& find_job(const DDBatch& B, int& local)
{
    int jb = 0;
    for (int k = 1; k < B.n; ++k)
        if ((int)blockIdx.x >= B.job[k].blockStart) jb = k;
    local = (int)blockIdx.x - B.job[jb].blockStart;
    return B.job[jb];
}

// s_waitcnt bounding only the vector memory counter (gfx9 encoding:
// vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits 15:14; expcnt and lgkmcnt at
// their maxima, i.e. not waited for).
template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    static_assert(N >= 0 && N < 64, "vmcnt out of range");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

__device__ __forceinline__ void bare_barrier() { asm volatile("s_barrier" ::: "memory"); }

// A barrier after this wave's LDS writes have landed.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// LDS address (byte offset in the workgroup's LDS) of a __shared__ pointer.
__device__ __forceinline__ uint32_t lds_addr(const void* p)
{
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

}  // namespace ppl
