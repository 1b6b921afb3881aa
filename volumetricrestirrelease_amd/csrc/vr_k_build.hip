// vr_k_build.hip -- volume grids built on the GPU from dense device grids: the
// same mip and conservative grids, brick tables, occupancy words, apron pools and
// bounds that the host build (vr_volume.cpp) makes, value for value, so that a
// frame of an animated volume can be rebuilt every frame without a trip through
// host memory.
//
// Every kernel repeats the host build's arithmetic in the host build's order
// (2x box reduction summed x-major, the 27-neighbourhood mean of the conservative
// grid, the tiny-value clamp against the grid maximum, round-to-nearest-even
// fp16, and a brick's bounds summed over its 10^3 apron with x outermost), so a
// device-built slot equals the host-built slot byte for byte.
//
// HBM bounds a large build, launches and waits a small one. The dense grid is read
// once for everything that is not a brick (kLevels: both mip chains and the largest
// value of every brick of every level), the full-resolution clamped and dilated
// grids are never stored (the fills of their occupied bricks form those values again),
// the tables of all slots come from four launches together, and one wait for the
// brick counts serves them all. 1024^3 with temperature, 4 mips, fp16: 31.6 -> 5.35 ms
// against a pass per step and a wait per slot (kLevels 2.5 ms, of which reading the grid
// once takes 0.7, the temperature's kBrickMax 0.74 = 5.8 TB/s, the fills 1.7: their
// VALU work per value); 96^3, 3 mips: 1.72 -> 0.15 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>

#include "vr_launch.h"
#include "vr_volume.h"

namespace vr {

namespace {

constexpr int kBuildThreads = 256;

__device__ __forceinline__ size_t lin(int x, int y, int z, int nx, int ny) {
    return (size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * (size_t)z);
}
// A raw grid's value as the build takes it (negative and NaN to 0), 0 outside the grid.
__device__ __forceinline__ float at(const float* __restrict__ s, int x, int y, int z, int nx, int ny, int nz) {
    if (x < 0 || y < 0 || z < 0 || x >= nx || y >= ny || z >= nz) return 0.f;
    const float v = s[lin(x, y, z, nx, ny)];
    return v > 0.f ? v : 0.f;
}

// IEEE binary16 bits of a float, round to nearest even (the host build's rule,
// written on the bits so that no device conversion mode can differ from it).
__device__ __forceinline__ uint16_t halfBits(float f) {
    const uint32_t x = __float_as_uint(f);
    const uint32_t sign = (x >> 16) & 0x8000u;
    const uint32_t absx = x & 0x7FFFFFFFu;
    if (absx >= 0x7F800000u) return (uint16_t)(sign | (absx > 0x7F800000u ? 0x7E00u : 0x7C00u));
    if (absx >= 0x477FF000u) return (uint16_t)(sign | 0x7C00u);
    if (absx < 0x38800000u) {
        if (absx < 0x33000000u) return (uint16_t)sign;
        const uint32_t mant = (absx & 0x7FFFFFu) | 0x800000u;
        const int e = (int)(absx >> 23);
        const int shift = 126 - e;
        uint32_t hm = mant >> shift;
        const uint32_t rem = mant & ((1u << shift) - 1u);
        const uint32_t half = 1u << (shift - 1);
        if (rem > half || (rem == half && (hm & 1u))) hm++;
        return (uint16_t)(sign | hm);
    }
    uint32_t h = (((absx >> 23) - 112u) << 10) | ((absx >> 13) & 0x3FFu);
    const uint32_t rem = absx & 0x1FFFu;
    if (rem > 0x1000u || (rem == 0x1000u && (h & 1u))) h++;
    return (uint16_t)(sign | h);
}
__device__ __forceinline__ float halfValue(uint16_t h) {
    const uint32_t sign = (uint32_t)(h & 0x8000u) << 16;
    const uint32_t e = (h >> 10) & 0x1Fu, m = h & 0x3FFu;
    uint32_t x;
    if (e == 0) {
        if (m == 0) return __uint_as_float(sign);
        return __uint_as_float(__float_as_uint(ldexpf((float)m, -24)) | sign);
    }
    if (e == 31) x = sign | 0x7F800000u | (m << 13);
    else x = sign | ((e + 112u) << 23) | (m << 13);
    return __uint_as_float(x);
}
// The stored value of a raw value (values below 1e-9 of the grid maximum are 0).
__device__ __forceinline__ float stored(float x, float gmax, int fp16) {
    x = (gmax > 0.f && x / gmax < 1e-9f) ? 0.f : x;
    if (gmax <= 0.f) x = 0.f;
    return fp16 ? halfValue(halfBits(x)) : x;
}

__device__ __forceinline__ float laneMax(float m, int from, int to) {
    for (int o = from; o <= to; o <<= 1) m = fmaxf(m, __shfl_xor(m, o));
    return m;
}
// values are >= 0, so their bits order as the values do
__device__ __forceinline__ void maxInto(unsigned* __restrict__ bits, float m) {
    if (m > 0.f) atomicMax(bits, __float_as_uint(m));
}
// A voxel of the conservative grid: an empty voxel takes the mean of the positive
// values of its 27-neighbourhood, summed x outermost. t: the value at an offset (>= 0).
template <class T>
__device__ __forceinline__ float dilated(float v, T t) {
    if (v != 0.f) return v;
    float avg = 0.f;
    for (int ii = -1; ii <= 1; ii++)
        for (int jj = -1; jj <= 1; jj++)
            for (int kk = -1; kk <= 1; kk++) avg += t(ii, jj, kk);
    avg /= 27.f;
    return avg > 0.f ? avg : v;
}
// 2x box reduction, weight 1/8 per tap summed x-major, negative results to 0
template <class T>
__device__ __forceinline__ float reduced(T t) {
    float res = 0.f;
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++)
            for (int c = 0; c < 2; c++) res = __fadd_rn(res, __fmul_rn(0.125f, t(a, b, c)));
    return res > 0.f ? res : 0.f;
}

__global__ __launch_bounds__(kBuildThreads) void kClear(unsigned* __restrict__ p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0u;
}

// Both mip chains down to level 3 from one read of the raw grid. A workgroup takes a
// 64 x 8 x 8 tile (8 whole bricks of mip 0, one voxel row of level 3) and its
// one-voxel halo through LDS: the density and its dilation are formed there, reduced
// level by level, and each level's values and bricks' largest values written. A tile
// without a positive value (most of a sparse volume) writes its zeros and ends.
// Tiles wider in x than the 128-byte lines they touch, 8 deep so that level 3 and the
// bricks need no exchange between workgroups; 50 KB of LDS, three workgroups per CU.
constexpr int kTX = 64, kTY = 8, kTZ = 8;
constexpr int kRow = 72;  // LDS row: voxel x at 4 + x, so that 16-byte stores align
struct LevelGrids {
    float* out[2][4];         // level 1..3 grids of the density [0] and its dilation [1]
    unsigned* brickMax[2][4]; // level 0..3: the largest value (bits) per brick
};
template <bool ALIGNED>
__global__ __launch_bounds__(kBuildThreads) void kLevels(const float* __restrict__ s, int nx, int ny, int nz, int levels,
                                                         LevelGrids L, int* __restrict__ bad) {
    __shared__ __align__(16) float t[kTZ + 2][kTY + 2][kRow];
    __shared__ float dil[kTZ][kTY][kTX];
    __shared__ float m1[2][4][4][32], m2[2][2][2][16];
    __shared__ float part[2][4][8];
    const int x0 = (int)blockIdx.x * kTX, y0 = (int)blockIdx.y * kTY, z0 = (int)blockIdx.z * kTZ;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    bool positive = false, finite = true;
    // all of a thread's loads are issued before the first is used: 3 workgroups per CU
    // hold too few waves to cover HBM's latency otherwise (3.4 -> 2.5 ms at 1024^3)
    constexpr int kLoads = ((kTZ + 2) * (kTY + 2) * 16 + kBuildThreads - 1) / kBuildThreads;
    float v[kLoads][4];
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        const int i = tid + j * kBuildThreads, q = i & 15, r = i >> 4, ly = r % (kTY + 2), lz = r / (kTY + 2);
        const int x = x0 + 4 * q, y = y0 + ly - 1, z = z0 + lz - 1;
#pragma unroll
        for (int k = 0; k < 4; k++) v[j][k] = 0.f;
        if (lz < kTZ + 2 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz) {
            const float* src = s + lin(x, y, z, nx, ny);
            if (ALIGNED) {
                const float4 w = *reinterpret_cast<const float4*>(src);
                v[j][0] = w.x; v[j][1] = w.y; v[j][2] = w.z; v[j][3] = w.w;
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) v[j][k] = src[k];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        const int i = tid + j * kBuildThreads, q = i & 15, r = i >> 4, ly = r % (kTY + 2), lz = r / (kTY + 2);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            finite = finite && isfinite(v[j][k]);
            v[j][k] = v[j][k] > 0.f ? v[j][k] : 0.f;
            positive = positive || v[j][k] > 0.f;
        }
        if (lz < kTZ + 2)
            *reinterpret_cast<float4*>(&t[lz][ly][4 + 4 * q]) = make_float4(v[j][0], v[j][1], v[j][2], v[j][3]);
    }
    if (tid < 2 * (kTZ + 2) * (kTY + 2)) {
        const int e = tid & 1, r = tid >> 1, ly = r % (kTY + 2), lz = r / (kTY + 2);
        const float v = at(s, e ? x0 + kTX : x0 - 1, y0 + ly - 1, z0 + lz - 1, nx, ny, nz);
        positive = positive || v > 0.f;
        t[lz][ly][e ? 4 + kTX : 3] = v;
    }
    if (!finite) *bad = 1;
    const int any = __syncthreads_or(positive ? 1 : 0);
    const int nbx = nx / 8, nby = ny / 8, bricks = min(8, nbx - 8 * (int)blockIdx.x);
    const size_t b0 = 8 * (size_t)blockIdx.x + (size_t)nbx * (blockIdx.y + (size_t)nby * blockIdx.z);
    if (!any) {
        if (tid < 2 * bricks) L.brickMax[tid / bricks][0][b0 + tid % bricks] = 0u;
        for (int l = 1; l <= levels; l++) {
            const int w = kTX >> l, h = kTY >> l, n = w * h * (kTZ >> l), gx = nx >> l, gy = ny >> l;
            for (int i = tid; i < 2 * n; i += kBuildThreads) {
                const int c = i / n, j = i % n, x = (x0 >> l) + j % w, y = (y0 >> l) + j / w % h, z = (z0 >> l) + j / w / h;
                if (x < gx) L.out[c][l][lin(x, y, z, gx, gy)] = 0.f;
            }
        }
        return;
    }
    // level 0: the dilation, and the largest value of each of the tile's bricks (8 lanes wide each)
    float md = 0.f, mc = 0.f;
    for (int r = wv; r < kTY * kTZ; r += 4) {
        const int y = r % kTY, z = r / kTY;
        const float v = t[z + 1][y + 1][4 + lane];
        const float c = dilated(v, [&](int i, int j, int k) { return t[z + 1 + k][y + 1 + j][4 + lane + i]; });
        dil[z][y][lane] = c;
        md = fmaxf(md, v);
        mc = fmaxf(mc, c);
    }
    md = laneMax(md, 1, 4);
    mc = laneMax(mc, 1, 4);
    if ((lane & 7) == 0) { part[0][wv][lane >> 3] = md; part[1][wv][lane >> 3] = mc; }
    __syncthreads();
    if (tid < 16) {
        const int c = tid >> 3, b = tid & 7;
        const float m = fmaxf(fmaxf(part[c][0][b], part[c][1][b]), fmaxf(part[c][2][b], part[c][3][b]));
        if (b < bricks) L.brickMax[c][0][b0 + b] = __float_as_uint(m);
    }
    if (levels < 1) return;
    // level l's bricks cover 2^l tiles a side in y and z: their maxima meet in memory
    auto brickAtLevel = [&](int l, int bx) {
        const int bw = (nx >> l) / 8, bh = (ny >> l) / 8;
        return (size_t)bx + (size_t)bw * (size_t)(((y0 >> l) / 8) + (size_t)bh * ((z0 >> l) / 8));
    };
    {
        const int gx = nx >> 1, gy = ny >> 1;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            float m = 0.f;
            for (int r = wv * 2 + (lane >> 5); r < 16; r += 8) {
                const int x = lane & 31, y = r & 3, z = r >> 2;
                const float o = c == 0 ? reduced([&](int a, int b, int k) { return t[2 * z + k + 1][2 * y + b + 1][4 + 2 * x + a]; })
                                       : reduced([&](int a, int b, int k) { return dil[2 * z + k][2 * y + b][2 * x + a]; });
                m1[c][z][y][x] = o;
                // voxels past the grid's edge are 0 and not stored
                if (x0 / 2 + x < gx) L.out[c][1][lin(x0 / 2 + x, y0 / 2 + y, z0 / 2 + z, gx, gy)] = o;
                if (x0 / 2 + x < gx) m = fmaxf(m, o);
            }
            m = laneMax(laneMax(m, 1, 4), 32, 32);
            if (lane < 32 && (lane & 7) == 0 && m > 0.f)
                maxInto(&L.brickMax[c][1][brickAtLevel(1, (x0 / 2 + lane) / 8)], m);
        }
    }
    if (levels < 2) return;
    __syncthreads();
    if (tid < 128) {
        const int c = wv, x = lane & 15, y = (lane >> 4) & 1, z = lane >> 5, gx = nx >> 2, gy = ny >> 2;
        float o = reduced([&](int a, int b, int k) { return m1[c][2 * z + k][2 * y + b][2 * x + a]; });
        m2[c][z][y][x] = o;
        const bool in = x0 / 4 + x < gx;
        if (in) L.out[c][2][lin(x0 / 4 + x, y0 / 4 + y, z0 / 4 + z, gx, gy)] = o;
        const float m = laneMax(laneMax(in ? o : 0.f, 1, 4), 16, 32);
        if (lane < 16 && (lane & 7) == 0) maxInto(&L.brickMax[c][2][brickAtLevel(2, min(x0 / 4 + x, gx - 1) / 8)], m);
    }
    if (levels < 3) return;
    __syncthreads();
    if (tid < 16) {
        const int c = tid >> 3, x = tid & 7, gx = nx >> 3, gy = ny >> 3;
        const float o = reduced([&](int a, int b, int k) { return m2[c][k][b][2 * x + a]; });
        if (x0 / 8 + x < gx) {
            L.out[c][3][lin(x0 / 8 + x, y0 / 8, z0 / 8, gx, gy)] = o;
            maxInto(&L.brickMax[c][3][brickAtLevel(3, (x0 / 8 + x) / 8)], o);
        }
    }
}

// The largest value of every brick of a grid (negative and NaN taken as 0); one
// workgroup per 64 x 8 x 8 tile. bad: set when a value is not finite.
template <bool ALIGNED>
__global__ __launch_bounds__(kBuildThreads) void kBrickMax(const float* __restrict__ s, int nx, int ny, int nz,
                                                           unsigned* __restrict__ brickMax, int* __restrict__ bad) {
    __shared__ float part[4][8];
    const int x0 = (int)blockIdx.x * kTX, y0 = (int)blockIdx.y * 8, z0 = (int)blockIdx.z * 8;
    const int q = threadIdx.x & 15, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    float m = 0.f;
    bool finite = true;
    if (x0 + 4 * q < nx) {
        float v[16];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = (threadIdx.x >> 4) + 16 * i;
            const float* src = s + lin(x0 + 4 * q, y0 + (r & 7), z0 + (r >> 3), nx, ny);
            if (ALIGNED) {
                const float4 w = *reinterpret_cast<const float4*>(src);
                v[4 * i] = w.x; v[4 * i + 1] = w.y; v[4 * i + 2] = w.z; v[4 * i + 3] = w.w;
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) v[4 * i + k] = src[k];
            }
        }
#pragma unroll
        for (int i = 0; i < 16; i++) {
            finite = finite && isfinite(v[i]);
            m = fmaxf(m, v[i] > 0.f ? v[i] : 0.f);
        }
    }
    if (!finite) *bad = 1;
    m = laneMax(laneMax(m, 1, 1), 16, 32);
    if (lane < 16 && (lane & 1) == 0) part[wv][lane >> 1] = m;
    __syncthreads();
    if (threadIdx.x < 8 && x0 + 8 * (int)threadIdx.x < nx) {
        const int b = threadIdx.x;
        m = fmaxf(fmaxf(part[0][b], part[1][b]), fmaxf(part[2][b], part[3][b]));
        brickMax[x0 / 8 + b + (size_t)(nx / 8) * (blockIdx.y + (size_t)(ny / 8) * blockIdx.z)] = __float_as_uint(m);
    }
}
// One 2x reduction of a whole grid (levels past kLevels'); d is nx/2 x ny/2 x nz/2
__global__ __launch_bounds__(kBuildThreads) void kReduce2(const float* __restrict__ s, float* __restrict__ d, int nx,
                                                          int ny, int nz) {
    const int dx = nx / 2, dy = ny / 2, dz = nz / 2;
    const size_t n = (size_t)dx * dy * dz;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % dx), y = (int)((i / dx) % dy), z = (int)(i / ((size_t)dx * dy));
        d[i] = reduced([&](int a, int b, int c) { return s[lin(2 * x + a, 2 * y + b, 2 * z + c, nx, ny)]; });
    }
}

// The tables of every slot of a frame, blockIdx.y = slot: the grid's largest value,
// the occupancy words, their prefix sums, the brick ids and the block table.
struct TableJobs {
    BuildGrid g[kFrameSlots];
    BuildStats* stats;
};
// Each step is a body over a range of threads (i of n), so that a frame of small grids can
// run all of them in one workgroup a slot (kTablesSmall) and a large one a launch each.
__device__ __forceinline__ float gridMaxBody(const BuildGrid& g, size_t i, size_t n) {
    float m = 0.f;
    for (size_t c = i; c < g.cells; c += n) m = fmaxf(m, __uint_as_float(g.brickMax[c]));
    return laneMax(m, 1, 32);
}
// Occupancy: does a brick hold a value that its stored form keeps above 0? Storing is
// monotone, so its largest value tells. Also clears the block and ahead tables.
__device__ __forceinline__ void wordsBody(const BuildGrid& g, float gmax, int fp16, size_t i, size_t n) {
    for (size_t k = i; k < g.blocks; k += n) g.nodes[k] = 0u;
    for (size_t k = i; k < kAheadBytes / 4; k += n) reinterpret_cast<uint32_t*>(g.ahead)[k] = 0u;
    // whole waves iterate together: 64 cells are two words
    for (size_t c = i; c - (threadIdx.x & 63) < g.cells; c += n) {
        const bool occ = c < g.cells && stored(__uint_as_float(g.brickMax[c]), gmax, fp16) > 0.f;
        const uint64_t bits = __ballot(occ);
        const int l = threadIdx.x & 63;
        if ((l & 31) == 0 && c < g.cells) g.words[2 * (c / 32)] = (uint32_t)(l ? bits >> 32 : bits);
    }
}
// Exclusive prefix of the words' popcounts into their second entries, one workgroup of
// 1024 a slot: 4096 consecutive words an iteration, scanned by wave and then across the
// waves. Returns the number of bricks.
__device__ __forceinline__ uint32_t scanBody(const BuildGrid& g, uint32_t* waveSum) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const size_t nw = (g.cells + 31) / 32;
    uint32_t base = 0u;
    for (size_t w0 = 0; w0 < nw; w0 += 4096) {
        const size_t w = w0 + 4 * threadIdx.x;
        uint32_t n[4], sum = 0u;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            n[k] = w + k < nw ? (uint32_t)__popc(g.words[2 * (w + k)]) : 0u;
            sum += n[k];
        }
        uint32_t incl = sum;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = (uint32_t)__shfl_up((int)incl, o);
            if (lane >= o) incl += y;
        }
        if (lane == 63) waveSum[wv] = incl;
        __syncthreads();
        uint32_t before = base, all = base;
        for (int k = 0; k < 16; k++) {
            if (k < wv) before += waveSum[k];
            all += waveSum[k];
        }
        before += incl - sum;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (w + k < nw) g.words[2 * (w + k) + 1] = before;
            before += n[k];
        }
        base = all;
        __syncthreads();
    }
    return base;
}
__device__ __forceinline__ void brickIdsBody(const BuildGrid& g, size_t i, size_t n) {
    const uint32_t nbx = g.nx / 8, nby = g.ny / 8;
    const int as = g.aheadShift;
    for (size_t c = i; c < g.cells; c += n) {
        const uint32_t bits = g.words[2 * (c / 32)], b = (uint32_t)(c % 32);
        if (!((bits >> b) & 1u)) { g.table[c] = kEmpty; continue; }
        const uint32_t id = g.words[2 * (c / 32) + 1] + (uint32_t)__popc(bits & ((1u << b) - 1u));
        g.table[c] = id;
        g.cellOf[id] = (uint32_t)c;
        const uint32_t r = (uint32_t)c / nbx, bx = (uint32_t)c % nbx, by = r % nby, bz = r / nby;
        g.nodes[(bx / 16) + (size_t)g.nnx * ((by / 16) + (size_t)g.nny * (bz / 16))] = 1u;
        g.ahead[(bx >> as) + (((nbx - 1) >> as) + 1) * ((by >> as) + (((nby - 1) >> as) + 1) * (bz >> as))] = 0xFFu;
    }
}
// The ahead table (Grid::ahead) from the groups that brickIdsBody marked: per axis, the
// octants that increase on it gather from the high side, the others from the low side; a
// thread a line.
__device__ __forceinline__ void aheadBody(const BuildGrid& g, uint8_t* t) {
    const int n[3] = {((g.nx / 8 - 1) >> g.aheadShift) + 1, ((g.ny / 8 - 1) >> g.aheadShift) + 1,
                      ((g.nz / 8 - 1) >> g.aheadShift) + 1};
    const int all = n[0] * n[1] * n[2], step[3] = {1, n[0], n[0] * n[1]};
    for (int i = threadIdx.x; i < all; i += blockDim.x) t[i] = g.ahead[i];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        __syncthreads();
        const int b = a == 0 ? 1 : 0, c = a == 2 ? 1 : 2;
        const uint32_t up = a == 0 ? 0xAAu : (a == 1 ? 0xCCu : 0xF0u);
        const int line = threadIdx.x;
        if (line < n[b] * n[c]) {
            uint8_t* l = t + (line % n[b]) * step[b] + (line / n[b]) * step[c];
            uint32_t v[kAheadSide], m = 0u;
#pragma unroll
            for (int i = 0; i < kAheadSide; i++) v[i] = i < n[a] ? l[i * step[a]] : 0u;
#pragma unroll
            for (int i = kAheadSide - 1; i >= 0; i--) m = (v[i] |= m) & up;
            m = 0u;
#pragma unroll
            for (int i = 0; i < kAheadSide; i++) m = (v[i] |= m) & ~up;
#pragma unroll
            for (int i = 0; i < kAheadSide; i++)
                if (i < n[a]) l[i * step[a]] = (uint8_t)v[i];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < all; i += blockDim.x) g.ahead[i] = t[i];
}

__global__ __launch_bounds__(kBuildThreads) void kGridMax(const TableJobs J) {
    const float m = gridMaxBody(J.g[blockIdx.y], (size_t)blockIdx.x * blockDim.x + threadIdx.x,
                                (size_t)gridDim.x * blockDim.x);
    if ((threadIdx.x & 63) == 0) maxInto(&J.stats->maxBits[blockIdx.y], m);
}
__global__ __launch_bounds__(kBuildThreads) void kWords(const TableJobs J, int fp16) {
    wordsBody(J.g[blockIdx.y], __uint_as_float(J.stats->maxBits[blockIdx.y]), fp16,
              (size_t)blockIdx.x * blockDim.x + threadIdx.x, (size_t)gridDim.x * blockDim.x);
}
__global__ __launch_bounds__(1024) void kScanWords(const TableJobs J) {
    __shared__ uint32_t waveSum[16];
    const uint32_t n = scanBody(J.g[blockIdx.y], waveSum);
    if (threadIdx.x == 0) J.stats->count[blockIdx.y] = n;
}
__global__ __launch_bounds__(kBuildThreads) void kBrickIds(const TableJobs J) {
    brickIdsBody(J.g[blockIdx.y], (size_t)blockIdx.x * blockDim.x + threadIdx.x, (size_t)gridDim.x * blockDim.x);
}
__global__ __launch_bounds__(kAheadSide* kAheadSide) void kAhead(const TableJobs J) {
    __shared__ uint8_t t[kAheadBytes];
    aheadBody(J.g[blockIdx.y], t);
}
// All of it for a slot in one workgroup, for grids of at most kSmallCells bricks: five
// launches' starts and gaps cost more than one workgroup's passes (a build of 96^3, 6
// slots: 0.185 -> 0.152 ms; at 256^3 a pass is 32 iterations).
constexpr size_t kSmallCells = 32768;
__global__ __launch_bounds__(1024) void kTablesSmall(const TableJobs J, int fp16) {
    const BuildGrid& g = J.g[blockIdx.y];
    __shared__ uint32_t waveSum[16];
    __shared__ float waveMax[16];
    __shared__ uint8_t t[kAheadBytes];
    const float m = gridMaxBody(g, threadIdx.x, 1024);
    if ((threadIdx.x & 63) == 0) waveMax[threadIdx.x >> 6] = m;
    __syncthreads();
    float gmax = 0.f;
    for (int k = 0; k < 16; k++) gmax = fmaxf(gmax, waveMax[k]);
    wordsBody(g, gmax, fp16, threadIdx.x, 1024);
    __syncthreads();
    const uint32_t n = scanBody(g, waveSum);
    if (threadIdx.x == 0) {
        J.stats->maxBits[blockIdx.y] = __float_as_uint(gmax);
        J.stats->count[blockIdx.y] = n;
    }
    __syncthreads();
    brickIdsBody(g, threadIdx.x, 1024);
    __syncthreads();
    aheadBody(g, t);
}

// Per brick its 10^3 apron values (stored form) and bounds {min, max, sum / 512, 0}.
// A wave fills a brick: 16 values a lane, rows of the source read along x. The
// bounds' sum runs over the apron with x outermost, one add after the other, as the
// host's: the values go through LDS in that order and one lane a brick adds them,
// 4 bricks side by side. DIL: the bricks of the dilated raw grid, whose values are
// formed from a 12^3 region in LDS.
struct FillJobs {
    int n;
    int start[kFrameSlots + 1];  // first workgroup of each slot
    uint32_t count[kFrameSlots];
    float least[kFrameSlots];    // the smallest value whose stored form is not clamped to 0
    BuildGrid g[kFrameSlots];
};
// The smallest x with x / gmax >= 1e-9 (stored()'s clamp; the quotient is monotone in x):
// a compare per value in place of a division.
float leastKept(float gmax) {
    if (!(gmax > 0.f)) return std::numeric_limits<float>::infinity();
    float x = 1e-9f * gmax;
    while (x > 0.f && x / gmax >= 1e-9f) x = std::nextafter(x, 0.f);
    while (x / gmax < 1e-9f) x = std::nextafter(x, gmax);
    return x;
}
constexpr int kFillBricks = 4, kFillRow = 1004;
template <int FP16, bool DIL>
__global__ __launch_bounds__(64 * kFillBricks) void kBrickFill(const FillJobs J) {
    __shared__ __align__(16) float vals[kFillBricks][kFillRow];
    __shared__ float raw[DIL ? kFillBricks : 1][DIL ? 1728 : 1];
    int i = 0;
    while (i + 1 < J.n && (int)blockIdx.x >= J.start[i + 1]) i++;
    const BuildGrid& g = J.g[i];
    const float least = J.least[i];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const size_t id0 = (size_t)((int)blockIdx.x - J.start[i]) * kFillBricks, id = id0 + wv;
    const bool live = id < J.count[i];
    const uint32_t nbx = g.nx / 8, nby = g.ny / 8, c = live ? g.cellOf[id] : 0u;
    const int x0 = (int)(c % nbx) * 8, y0 = (int)(c / nbx % nby) * 8, z0 = (int)(c / nbx / nby) * 8;
    if constexpr (DIL) {
        if (live) {
            float r[27];
#pragma unroll
            for (int k = 0; k < 27; k++) {
                const int v = lane + 64 * k;
                r[k] = at(g.src, x0 + v % 12 - 2, y0 + v / 12 % 12 - 2, z0 + v / 144 - 2, g.nx, g.ny, g.nz);
            }
#pragma unroll
            for (int k = 0; k < 27; k++) raw[wv][lane + 64 * k] = r[k];
        }
        __syncthreads();
    }
    float mn = 3.402823466e+38f, mx = 0.f;
    if (live) {
        // two neighbours along x a lane: one 4-byte store of an fp16 pair. The loads of all
        // of a lane's values are issued together
        constexpr int kPairs = (kBrickVals / 2 + 63) / 64;
        float r[kPairs][2];
#pragma unroll
        for (int j = 0; j < kPairs; j++) {
            const int v = 2 * lane + 128 * j, a = v % kApron, b = v / kApron % kApron, d = v / (kApron * kApron);
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int x = x0 + a + e - 1, y = y0 + b - 1, z = z0 + d - 1;
                if (v >= kBrickVals) r[j][e] = 0.f;
                else if constexpr (DIL) {
                    const bool in = x >= 0 && y >= 0 && z >= 0 && x < g.nx && y < g.ny && z < g.nz;
                    const float* t = &raw[wv][(a + e + 1) + 12 * ((b + 1) + 12 * (d + 1))];
                    r[j][e] = in ? dilated(t[0], [&](int ii, int jj, int kk) { return t[ii + 12 * (jj + 12 * kk)]; }) : 0.f;
                } else {
                    r[j][e] = at(g.src, x, y, z, g.nx, g.ny, g.nz);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < kPairs; j++) {
            const int v = 2 * lane + 128 * j, a = v % kApron, b = v / kApron % kApron, d = v / (kApron * kApron);
            if (v >= kBrickVals) continue;
            // stored() by the conversion unit: round to nearest even, overflow to infinity and
            // subnormals kept, as halfBits rounds (values here are finite and >= 0)
            float o[2];
            uint16_t hb[2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                o[e] = r[j][e] < least ? 0.f : r[j][e];
                if (FP16) {
                    const _Float16 h = (_Float16)o[e];
                    hb[e] = __builtin_bit_cast(uint16_t, h);
                    o[e] = (float)h;
                }
                vals[wv][(a + e) * 100 + b * 10 + d] = o[e];
                mn = fminf(mn, o[e]);
                mx = fmaxf(mx, o[e]);
            }
            if (FP16)
                reinterpret_cast<uint32_t*>((uint16_t*)g.pool + id * kBrickVals)[v / 2] =
                    (uint32_t)hb[0] | (uint32_t)hb[1] << 16;
            else
                reinterpret_cast<float2*>((float*)g.pool + id * kBrickVals)[v / 2] = make_float2(o[0], o[1]);
        }
        for (int o = 1; o < 64; o <<= 1) {
            mn = fminf(mn, __shfl_xor(mn, o));
            mx = fmaxf(mx, __shfl_xor(mx, o));
        }
        if (lane == 0) {
            g.bounds[4 * id + 0] = mn;
            g.bounds[4 * id + 1] = mx;
            g.bounds[4 * id + 3] = 0.f;
        }
    }
    __syncthreads();
    if (threadIdx.x < kFillBricks && id0 + threadIdx.x < J.count[i]) {
        const float4* v = reinterpret_cast<const float4*>(vals[threadIdx.x]);
        float sum = 0.f;
#pragma unroll 10
        for (int k = 0; k < kBrickVals / 4; k++) {
            const float4 q = v[k];
            sum = __fadd_rn(__fadd_rn(__fadd_rn(__fadd_rn(sum, q.x), q.y), q.z), q.w);
        }
        g.bounds[4 * (id0 + threadIdx.x) + 2] = sum / 512.f;
    }
}

dim3 gridFor(size_t n) { return dim3((unsigned)std::min<size_t>((n + kBuildThreads - 1) / kBuildThreads, 65536)); }
bool aligned16(const void* p) { return ((uintptr_t)p % 16) == 0; }
dim3 tileGrid(int nx, int ny, int nz) { return dim3((unsigned)((nx + kTX - 1) / kTX), (unsigned)(ny / 8), (unsigned)(nz / 8)); }

}  // namespace

hipError_t buildClear(hipStream_t st, void* p, size_t words) {
    hipLaunchKernelGGL(kClear, gridFor(words), dim3(kBuildThreads), 0, st, (unsigned*)p, words);
    return hipGetLastError();
}
hipError_t buildLevels(hipStream_t st, const float* s, int nx, int ny, int nz, int levels, float* const out[2][4],
                       unsigned* const brickMax[2][4], int* bad) {
    LevelGrids L;
    for (int c = 0; c < 2; c++)
        for (int l = 0; l < 4; l++) { L.out[c][l] = out[c][l]; L.brickMax[c][l] = brickMax[c][l]; }
    if (aligned16(s))
        hipLaunchKernelGGL(kLevels<true>, tileGrid(nx, ny, nz), dim3(kBuildThreads), 0, st, s, nx, ny, nz, levels, L, bad);
    else
        hipLaunchKernelGGL(kLevels<false>, tileGrid(nx, ny, nz), dim3(kBuildThreads), 0, st, s, nx, ny, nz, levels, L, bad);
    return hipGetLastError();
}
hipError_t buildBrickMax(hipStream_t st, const float* s, int nx, int ny, int nz, unsigned* brickMax, int* bad) {
    if (aligned16(s))
        hipLaunchKernelGGL(kBrickMax<true>, tileGrid(nx, ny, nz), dim3(kBuildThreads), 0, st, s, nx, ny, nz, brickMax, bad);
    else
        hipLaunchKernelGGL(kBrickMax<false>, tileGrid(nx, ny, nz), dim3(kBuildThreads), 0, st, s, nx, ny, nz, brickMax, bad);
    return hipGetLastError();
}
hipError_t buildReduce2(hipStream_t st, const float* s, float* d, int nx, int ny, int nz) {
    hipLaunchKernelGGL(kReduce2, gridFor((size_t)(nx / 2) * (ny / 2) * (nz / 2)), dim3(kBuildThreads), 0, st, s, d, nx,
                       ny, nz);
    return hipGetLastError();
}
hipError_t buildTables(hipStream_t st, const BuildGrid* grids, int n, bool fp16, BuildStats* stats) {
    if (n < 1 || n > kFrameSlots) return hipErrorInvalidValue;
    TableJobs J{};
    J.stats = stats;
    size_t cells = 0;
    for (int i = 0; i < n; i++) {
        J.g[i] = grids[i];
        cells = std::max(cells, grids[i].cells);
    }
    if (cells <= kSmallCells) {
        hipLaunchKernelGGL(kTablesSmall, dim3(1, n), dim3(1024), 0, st, J, fp16 ? 1 : 0);
        return hipGetLastError();
    }
    const dim3 g((unsigned)std::min<size_t>((cells + kBuildThreads - 1) / kBuildThreads, 512), n);
    hipLaunchKernelGGL(kGridMax, g, dim3(kBuildThreads), 0, st, J);
    hipLaunchKernelGGL(kWords, g, dim3(kBuildThreads), 0, st, J, fp16 ? 1 : 0);
    hipLaunchKernelGGL(kScanWords, dim3(1, n), dim3(1024), 0, st, J);
    hipLaunchKernelGGL(kBrickIds, g, dim3(kBuildThreads), 0, st, J);
    hipLaunchKernelGGL(kAhead, dim3(1, n), dim3(kAheadSide * kAheadSide), 0, st, J);
    return hipGetLastError();
}
hipError_t buildFill(hipStream_t st, const BuildGrid* grids, const BuildStats& stats, int n, bool fp16) {
    if (n < 1 || n > kFrameSlots) return hipErrorInvalidValue;
    for (int dil = 0; dil < 2; dil++) {
        FillJobs J{};
        for (int i = 0; i < n; i++) {
            if (grids[i].dilate != (dil != 0) || stats.count[i] == 0) continue;
            const int k = J.n++;
            J.g[k] = grids[i];
            J.count[k] = stats.count[i];
            float gmax;
            std::memcpy(&gmax, &stats.maxBits[i], 4);
            J.least[k] = leastKept(gmax);
            J.start[k + 1] = J.start[k] + (int)((stats.count[i] + kFillBricks - 1) / kFillBricks);
        }
        if (J.n == 0) continue;
        const dim3 g((unsigned)J.start[J.n]), blk(64 * kFillBricks);
        if (fp16 && dil) hipLaunchKernelGGL((kBrickFill<1, true>), g, blk, 0, st, J);
        else if (fp16) hipLaunchKernelGGL((kBrickFill<1, false>), g, blk, 0, st, J);
        else if (dil) hipLaunchKernelGGL((kBrickFill<0, true>), g, blk, 0, st, J);
        else hipLaunchKernelGGL((kBrickFill<0, false>), g, blk, 0, st, J);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
// The slot's descriptor once its buffers are filled (w2i is the caller's)
void buildDescribe(const BuildGrid& b, const BuildStats& stats, int i, bool fp16, Grid& G) {
    float gmax;
    std::memcpy(&gmax, &stats.maxBits[i], 4);
    // the stored form of the maximum (monotone, so the largest stored value)
    float mv = gmax;
    if (!(gmax > 0.f)) mv = 0.f;
    else if (fp16) mv = halfBitsToFloat(floatToHalfBits(gmax));
    std::memset(&G, 0, sizeof(Grid));
    G.brickTable = b.table;
    G.nodeTable = b.nodes;
    G.occ = b.words;
    G.occWords = (int32_t)((b.cells + 31) / 32);
    G.ahead = b.ahead;
    G.aheadShift = b.aheadShift;
    G.numBricks = stats.count[i];
    G.bounds = b.bounds;
    G.pool = b.pool;
    G.nbx = b.nx / 8; G.nby = b.ny / 8; G.nbz = b.nz / 8;
    G.nnx = b.nnx; G.nny = b.nny; G.nnz = b.nnz;
    G.bmax[0] = (float)b.nx; G.bmax[1] = (float)b.ny; G.bmax[2] = (float)b.nz;
    G.maxValue = mv;
    G.fp16 = fp16 ? 1 : 0;
    G.channels = 1;
    G.valid = 1;
}

}  // namespace vr
