// c3d_append.h -- worklists of cells and their appends through LDS.  Needs nothing but atomicAdd,
// __syncthreads, threadIdx and blockDim, so that it can be compiled on the host, with a thread
// for each wave, to check its barriers.
#pragma once

namespace c3d {

// The worklists of one pass generation: cells in the mixed mode's FP32-Hessian phase and
// cells on the FP64 path (every cell outside the mixed mode).  Slot s of a pass is
// Wm[s] for s < *nm, else Wf[s - *nm].
struct Lists {
    int *Wm, *Wf;
    int *nm, *nf;
};

__device__ __forceinline__ int list_cell(const Lists &L, int slot, int nWm)
{
    return slot < nWm ? L.Wm[slot] : L.Wf[slot - nWm];
}

__device__ __forceinline__ void list_append(const Lists &L, bool mixedPhase, int c)
{
    if (mixedPhase)
        L.Wm[atomicAdd(L.nm, 1)] = c;
    else
        L.Wf[atomicAdd(L.nf, 1)] = c;
}

// Appends of a block to the next pass's lists, gathered in LDS and flushed with one global
// atomic per list and batch (a global atomic per cell on one counter serialises at the L2).
// push: one lane per cell, at most perRound pushes between two flush() calls; flush:
// called by the whole block at a block-uniform point.  Waves may run at any pace between the
// barriers: no two of them may see different counts, or they would part at a barrier.
constexpr int kAggCap = 256;
struct BlockAppender {
    int *buf;   // LDS [2][kAggCap]
    int *cnt;   // LDS [2]
    int *base;  // LDS [2]
    __device__ __forceinline__ void init()
    {
        if (threadIdx.x < 2)
            cnt[threadIdx.x] = 0;
        __syncthreads();
    }
    __device__ __forceinline__ void push(bool mixedPhase, int c)
    {
        const int l = mixedPhase ? 0 : 1;
        buf[l * kAggCap + atomicAdd(&cnt[l], 1)] = c;
    }
    // after a barrier: flush if forced or if another round of pushes might overflow
    __device__ __forceinline__ void flush(const Lists &L, bool force, int perRound)
    {
        __syncthreads();
        const int c0 = cnt[0], c1 = cnt[1];
        __syncthreads();  // every wave has them before the next round's pushes change them
        if (!force && c0 <= kAggCap - perRound && c1 <= kAggCap - perRound)
            return;
        if (threadIdx.x == 0) {
            base[0] = c0 ? atomicAdd(L.nm, c0) : 0;
            base[1] = c1 ? atomicAdd(L.nf, c1) : 0;
        }
        __syncthreads();
        for (int t = threadIdx.x; t < c0; t += blockDim.x)
            L.Wm[base[0] + t] = buf[t];
        for (int t = threadIdx.x; t < c1; t += blockDim.x)
            L.Wf[base[1] + t] = buf[kAggCap + t];
        __syncthreads();
        if (threadIdx.x < 2)
            cnt[threadIdx.x] = 0;
        __syncthreads();
    }
};

#define C3D_BLOCK_APPENDER(name)                                                          \
    __shared__ int name##_buf[2 * kAggCap];                                                \
    __shared__ int name##_cnt[2];                                                          \
    __shared__ int name##_base[2];                                                         \
    BlockAppender name{name##_buf, name##_cnt, name##_base};                               \
    name.init()

}  // namespace c3d
