// vr_segment.hpp -- how many samples a march takes in one brick, without marching it.
// Plain float arithmetic on scalars: the device march (vr_k_queue.hip) includes it, and a
// host build of it is compared with the loop on the CPU.
#pragma once
#include <math.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define VR_SEG_FN __host__ __device__ __forceinline__
#else
#define VR_SEG_FN static inline
#endif

namespace vr {

// The loop whose iterations are counted (TrMarch's brick loop without its samples): up to
// 128 samples at q, q + dq, ... (brick-local, each sum rounded) while inside the brick
// [0, 8)^3 and before tFar.
VR_SEG_FN int segmentLoop(float t, float qx, float qy, float qz, float dx, float dy, float dz, float tStep, float tFar) {
    int n = 0;
    while (n < 128 && qx >= 0.f && qy >= 0.f && qz >= 0.f && qx < 8.f && qy < 8.f && qz < 8.f && t < tFar) {
        qx += dx; qy += dy; qz += dz;
        t += tStep;
        n++;
    }
    return n;
}

// The count from a guess (r: steps until the ray leaves the brick or passes tFar, as the
// walk knows them), taken only when it is certain to be the loop's: sample n - 1 must lie
// inside the brick and before tFar, and sample n outside it or past tFar, by more than the
// loop's rounding can move them. Each of k additions rounds a coordinate of at most 8 by
// half an ulp, 2.4e-7, and the time by 6e-8 of its size; the last step out of the brick
// rounds by 6e-8 of where it lands, the step itself by 6e-8 of 8 over all of them, and
// forming the samples here costs as much again: the margins are these sums, rounded up.
// Positions move one way on each axis, so the samples between the first and the last are
// inside too. Everything else (rays that graze a face, times within rounding of tFar, 128
// samples, NaN) gives -1 and the loop tells: 2e-4 to 3e-3 of the segments with a sample at
// 0.2 to 2 voxels a step. Where the guess comes from does not matter for the result: the
// walk's exit time carries the rounding of grid coordinates divided by the direction, up to
// several steps for rays that graze a face, so a bound on the time alone will not do.
VR_SEG_FN int segmentCertain(float r, float t0, float qx, float qy, float qz, float dx, float dy, float dz,
                             float tStep, float tFar) {
    const bool first = qx >= 0.f && qy >= 0.f && qz >= 0.f && qx < 8.f && qy < 8.f && qz < 8.f;
    if (!(first && t0 < tFar)) return 0;
    const float nf = ceilf(r);
    if (!(nf >= 1.f && nf < 128.f)) return -1;
    const float k = nf - 1.f, m = 3e-7f * (nf + 3.f);
    const float tm = 8e-8f * (nf + 1.f) * (fabsf(t0) + nf * tStep);
    const float lx = fmaf(k, dx, qx), ly = fmaf(k, dy, qy), lz = fmaf(k, dz, qz), tl = fmaf(k, tStep, t0);
    const float lo = fminf(fminf(lx, ly), lz), hi = fmaxf(fmaxf(lx, ly), lz);
    const bool last = lo >= m && hi < 8.f - m && tl + tm < tFar;
    const float ox = lx + dx, oy = ly + dy, oz = lz + dz, sum = ox + oy + oz;
    const float low = fminf(fminf(ox, oy), oz), high = fmaxf(fmaxf(ox, oy), oz);
    const bool past = high - 8.f > m + 2e-7f * high || -low > m - 2e-7f * low || tl + tStep - tm >= tFar;
    return last && past && sum == sum ? (int)nf : -1;  // (min and max pass a NaN axis over)
}
VR_SEG_FN int segmentCount(float r, float t0, float qx, float qy, float qz, float dx, float dy, float dz, float tStep,
                           float tFar) {
    const int n = segmentCertain(r, t0, qx, qy, qz, dx, dy, dz, tStep, tFar);
    return n >= 0 ? n : segmentLoop(t0, qx, qy, qz, dx, dy, dz, tStep, tFar);
}

}  // namespace vr
