// Batched step kernels for the shot server on gfx950.
//
// One launch advances several stride-0 shots of the same radius by one time
// step each: the blocks of the launch are the shots' own receiver and step
// grids laid end to end, and every block finds its shot by a search over the prefix
// of block counts (kernel arguments), then runs the single-shot block body
// (step3d_z_block / step2d_z_block / receivers_block) on that shot's
// arrays with its step number.  Same operations per point as the
// single-shot kernels, so a batched shot gives the same bits as it alone.
// Slots follow the stride-0 cycle of the reference's time loop
// (wave.c:112-124): step n reads levels n-1 (slot (n-1) mod 3) and n (slot
// n mod 3) and writes level n+1 (slot (n+1) mod 3); its receivers read
// level n into row n-1 of the shot record.
#pragma once
#include "sw_kernels.hpp"

namespace sw {

// One shot's constants for batched launches, kept on the device by its plan.
struct BatchShot {
    Params P;                  // run constants (no graph step base)
    LapDiv D;                  // Laplacian quotient divisors (3D)
    real_t *u;                 // the three wavefield slots
    real_t *rec;               // shot record [steps][nrec]
    const Box *rbox;
    const real_t *rw;
    long long npts;            // slot stride (points)
    int nrec, nrb;             // receivers and their blocks, ahead of the step's
    int zlen;                  // z chunk of the step grid
    int gx, gy;                // step grid: blocks along the contiguous axis, then x
};

constexpr int kMaxBatch = 48;

#if SW_DIM == 3
constexpr int kBatchLines = kZLines, kRecPerBatch = kRecPerZ;
typedef RecZ RecBatch;
#else
constexpr int kBatchLines = 4, kRecPerBatch = sizeof(real_t) == 4 ? 16 : 8;
typedef RecShared<kRecPerBatch, 128> RecBatch;
#endif

// Arguments of one batched launch (by value): the shots, their step numbers
// and the first block of each (first[count] = blocks of the launch).
struct BatchArgs {
    const BatchShot *shot[kMaxBatch];
    int n[kMaxBatch];
    int first[kMaxBatch + 1];
    int count;
};

__device__ __forceinline__ int batch_shot(const BatchArgs &A, int b)
{
    int lo = 0, hi = A.count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (A.first[mid] <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

template <int R>
#if SW_DIM == 3
__global__ void __launch_bounds__(64 * kZLines, z_waves(R))
k_step3d_z_batch(BatchArgs A)
#else
__global__ void __launch_bounds__(kZ2Block)
k_step2d_z_batch(BatchArgs A)
#endif
{
    constexpr int NT = SW_DIM == 3 ? 64 * kBatchLines : 256;
    __shared__ RecBatch sh;
    const int s = batch_shot(A, blockIdx.x);
    const BatchShot *__restrict__ b = A.shot[s];
    const Params P = b->P;
    const int n = A.n[s];
    int local = blockIdx.x - A.first[s];
    const long long np = b->npts;
    real_t *u = b->u;
    const real_t *uc = u + (long long)(n % 3) * np;
    if (local < b->nrb) {
        receivers_beside<NT, R>(P, sh, uc, b->rbox, b->rw, b->nrec,
                                b->rec + (long long)(n - 1) * b->nrec, local,
                                SW_DIM == 3 ? threadIdx.y * 64 + threadIdx.x : threadIdx.x);
        return;
    }
    local -= b->nrb;
    const int gx = b->gx;
    const real_t *up = u + (long long)((n - 1) % 3) * np;
    real_t *un = u + (long long)((n + 1) % 3) * np;
#if SW_DIM == 3
    const LapDiv D = b->D;
    const int gy = b->gy, t = local / gx;
    step3d_z_block<R>(P, D, uc, up, un, n, b->zlen, local % gx, t % gy, t / gy);
#else
    step2d_z_block<R>(P, uc, up, un, n, b->zlen, local % gx, local / gx);
#endif
}

}  // namespace sw
