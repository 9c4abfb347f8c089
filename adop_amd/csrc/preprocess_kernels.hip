// preprocess_kernels.hip — point-cloud preprocessing that decides how well the rasterizer runs (gfx950): the distance
// of every point to its n-th nearest neighbour (SceneData::ComputeRadius, SceneData.cpp:441-484: a kd-tree
// k-nearest-neighbour search per point on the host) and the Morton code of every point (the key of ReorderMorton64,
// SceneData.cpp:101).
//
// Nearest neighbours: the points are put into the cells of a uniform grid, stored cell after cell, and every point
// then walks the cube of cells around its own until the n-th best distance cannot be beaten from outside the cube.
// The distances are formed as sqrt((dx*dx + dy*dy) + dz*dz) in fp32; the result is the n-th smallest of them over all
// other points, whatever the search order and whatever the grid, so a brute-force search over the same arithmetic
// gives the same bits. The cost is the number of candidates, which the cell size decides, and the right cell size
// depends on how the cloud fills space (scans are surfaces: a grid sized by volume puts hundreds of points into the
// few cells that have any). So the search grid is sized on the device (no host round trip) from the neighbour
// distances of 1024 sample points, measured in a part of the cloud (every 16th point) on a coarse grid sized by
// volume.  The coarse grid over the whole cloud is built only when the search grid leaves points undecided (sparse
// parts of the cloud), which the device finds out.
#include "cloud_kernels.h"
#include "common.h"
#include "launch.h"

#pragma clang fp contract(off)

namespace adop
{
// The search grid is stored in bricks of 8 x 4 x 4 cells: the points brick after brick and, inside a brick, cell
// after cell with x fastest.  A cloud of 10 M points asks for 100 M cells and more, nearly all of them empty: the
// bricks are counted in one dense table (a 128th of the cells) and only the bricks that hold points have a row in the
// table of the cells' first points.  (A dense table of cells took 650 us to clear and sum up for 10 M points on 1000
// patches, and its 10 M atomics on single cells 720 us; the bricks and the sort inside them take 235 us in all.)  A
// wavefront of consecutive points stays inside a brick or two, and so do the cells it searches.
constexpr int kBrickX = 3, kBrickY = 2, kBrickZ = 2;  // log2 of the cells per brick
static_assert(kBrickX + kBrickY + kBrickZ == 7 && (1 << 7) == kBrickCells, "128 cells");
constexpr uint32_t kNoBrick = 0xFFFFFFFFu;

// Cell of a point; points outside the grid's box (the box leaves the far tails of the cloud out) belong to the nearest
// boundary cell.
__device__ __forceinline__ int3 grid_cell(const KnnGrid& g, float x, float y, float z)
{
    const float fx = fminf(fmaxf((x - g.min[0]) * g.inv_cell, 0.f), (float)(g.dim[0] - 1));
    const float fy = fminf(fmaxf((y - g.min[1]) * g.inv_cell, 0.f), (float)(g.dim[1] - 1));
    const float fz = fminf(fmaxf((z - g.min[2]) * g.inv_cell, 0.f), (float)(g.dim[2] - 1));
    return make_int3((int)fx, (int)fy, (int)fz);
}

__device__ __forceinline__ uint32_t grid_index(const KnnGrid& g, int cx, int cy, int cz)
{
    return ((uint32_t)cz * (uint32_t)g.dim[1] + (uint32_t)cy) * (uint32_t)g.dim[0] + (uint32_t)cx;
}

// first brick of the row of bricks that holds the cells (., cy, cz); brick of cell cx: + (cx >> kBrickX)
__device__ __forceinline__ uint32_t brick_row(const KnnGrid& g, int cy, int cz)
{
    return ((uint32_t)(cz >> kBrickZ) * (uint32_t)g.bricks_y + (uint32_t)(cy >> kBrickY)) * (uint32_t)g.bricks_x;
}
__device__ __forceinline__ uint32_t brick_local(int cx, int cy, int cz)
{
    return (uint32_t)(cz & 3) << (kBrickX + kBrickY) | (uint32_t)(cy & 3) << kBrickX | (uint32_t)(cx & 7);
}
static_assert(kBrickY == 2 && kBrickZ == 2 && kBrickX == 3, "masks of brick_local");

// The points [first, end) of the cells xa..xb of row (cy, cz) of the brick in `slot` (xa and xb lie in that brick; a
// longer row is taken brick by brick).
__device__ __forceinline__ void brick_range(const KnnView& k, uint32_t slot, int xa, int xb, int cy, int cz,
                                            uint32_t* first, uint32_t* end)
{
    const uint32_t* row = k.cell_start + ((size_t)slot << 7) + brick_local(0, cy, cz);
    *first              = row[xa & 7];
    *end                = row[(xb & 7) + 1];
}

// ---- binning ----------------------------------------------------------------------------------------------------
// Points per bin (BRICKS: bricks of the search grid, else cells of the coarse grid) and the rank of every point in its
// bin.  Neighbouring lanes mostly hold points of one bin where the cloud is stored in spatial order: every run of equal
// bins takes its ranks with one returning atomic.  `stride` > 1: every stride-th point only (n of them).
constexpr int kBinPer = 4;

template <bool BRICKS>
__global__ __launch_bounds__(kBlock) void knn_count_kernel(const float4* __restrict__ position, int n, int stride,
                                                           const KnnGrid* __restrict__ gp, uint32_t* __restrict__ count,
                                                           uint32_t* __restrict__ rank, const uint32_t* __restrict__ gate)
{
    if (gate && *gate == 0) return;  // (kernel-uniform)
    const KnnGrid g    = *gp;
    const int lane     = threadIdx.x & 63;
    const size_t base  = (size_t)blockIdx.x * (kBlock * kBinPer) + threadIdx.x;
    float4 p[kBinPer];
#pragma unroll
    for (int k = 0; k < kBinPer; ++k)
    {
        const size_t i = base + k * kBlock;
        p[k]           = i < (size_t)n ? position[i * (size_t)stride] : make_float4(0, 0, 0, 0);
    }
    uint32_t first[kBinPer];
    int head[kBinPer];
#pragma unroll
    for (int k = 0; k < kBinPer; ++k)
    {
        const bool valid = base + k * kBlock < (size_t)n;
        const int3 c     = grid_cell(g, p[k].x, p[k].y, p[k].z);
        uint32_t b       = kNoBrick;
        if (valid) b = BRICKS ? brick_row(g, c.y, c.z) + (uint32_t)(c.x >> kBrickX) : grid_index(g, c.x, c.y, c.z);
        const uint32_t prev = (uint32_t)__shfl_up((int)b, 1, 64);
        const bool starts   = lane == 0 || prev != b;
        const unsigned long long heads = __ballot(starts);
        const unsigned long long upto  = (2ull << lane) - 1ull;  // lanes 0..lane (lane 63: all)
        head[k]  = 63 - __clzll((long long)(heads & upto));
        first[k] = 0;
        if (starts && valid)
        {
            const unsigned long long above = heads & ~upto;
            const int next                 = above ? __ffsll((long long)above) - 1 : 64;
            first[k]                       = atomicAdd(&count[b], (uint32_t)(next - lane));
        }
    }
#pragma unroll
    for (int k = 0; k < kBinPer; ++k)
    {
        const uint32_t f = (uint32_t)__shfl((int)first[k], head[k], 64);
        const size_t i   = base + k * kBlock;
        if (i < (size_t)n) __builtin_nontemporal_store(f + (uint32_t)(lane - head[k]), rank + i);
    }
}

// The points bin after bin, (x, y, z, bits of the point id): no atomics, the rank comes from the counting pass.
template <bool BRICKS>
__global__ __launch_bounds__(kBlock) void knn_scatter_kernel(const float4* __restrict__ position, int n, int stride,
                                                             const KnnGrid* __restrict__ gp,
                                                             const uint32_t* __restrict__ start,
                                                             const uint32_t* __restrict__ rank, float4* __restrict__ out,
                                                             const uint32_t* __restrict__ gate)
{
    if (gate && *gate == 0) return;
    const KnnGrid g   = *gp;
    const size_t base = (size_t)blockIdx.x * (kBlock * kBinPer) + threadIdx.x;
    float4 p[kBinPer];
    uint32_t r[kBinPer];
#pragma unroll
    for (int k = 0; k < kBinPer; ++k)
    {
        const size_t i = base + k * kBlock;
        p[k]           = i < (size_t)n ? position[i * (size_t)stride] : make_float4(0, 0, 0, 0);
        r[k]           = i < (size_t)n ? __builtin_nontemporal_load(rank + i) : 0u;
    }
#pragma unroll
    for (int k = 0; k < kBinPer; ++k)
    {
        const size_t i = base + k * kBlock;
        if (i >= (size_t)n) continue;
        const int3 c     = grid_cell(g, p[k].x, p[k].y, p[k].z);
        const uint32_t b = BRICKS ? brick_row(g, c.y, c.z) + (uint32_t)(c.x >> kBrickX) : grid_index(g, c.x, c.y, c.z);
        out[start[b] + r[k]] = make_float4(p[k].x, p[k].y, p[k].z, __uint_as_float((uint32_t)(i * (size_t)stride)));
    }
}

// Zeroes the counters of the grid's bins.
template <bool BRICKS>
__global__ __launch_bounds__(kBlock) void knn_clear_kernel(uint32_t* __restrict__ count, const KnnGrid* __restrict__ gp,
                                                           const uint32_t* __restrict__ gate)
{
    if (gate && *gate == 0) return;
    const uint32_t bins = BRICKS ? gp->bricks : gp->cells;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < bins; i += (size_t)gridDim.x * kBlock)
        __builtin_nontemporal_store(0u, count + i);
}

// Exclusive prefix sums over the bins in two launches: sums of chunks of 8192 bins, then the sums inside every chunk
// on top of those of the chunks before it (at most 1024 chunks, which every workgroup sums up for itself).  BRICKS:
// the bins that hold points are numbered in the same pass (slots), in the high half of a 64-bit sum.
constexpr int kScanChunk  = 8192;
constexpr int kScanChunks = 1024;

__device__ __forceinline__ unsigned long long block_exclusive_scan_1024(unsigned long long sum, unsigned long long* s_wave,
                                                                        unsigned long long* total)
{
    const int tid          = threadIdx.x;
    unsigned long long inc = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1)
    {
        const unsigned long long u = __shfl_up(inc, off, 64);
        if ((tid & 63) >= off) inc += u;
    }
    __syncthreads();  // s_wave of the last call has been read
    if ((tid & 63) == 63) s_wave[tid >> 6] = inc;
    __syncthreads();
    unsigned long long run = inc - sum, all = 0;
    for (int w = 0; w < 16; ++w)
    {
        if (w < (tid >> 6)) run += s_wave[w];
        all += s_wave[w];
    }
    *total = all;
    return run;
}

__device__ __forceinline__ void scan_load(const uint32_t* __restrict__ count, size_t t0, uint32_t bins, uint32_t v[8])
{
    if (t0 + 8 <= bins)
    {
        const uint4 a = ((const uint4*)(count + t0))[0], c = ((const uint4*)(count + t0))[1];
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = c.x, v[5] = c.y, v[6] = c.z, v[7] = c.w;
    }
    else
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = t0 + k < bins ? count[t0 + k] : 0u;
}

template <bool BRICKS>
__global__ __launch_bounds__(1024) void knn_scan_reduce_kernel(const uint32_t* __restrict__ count,
                                                               const KnnGrid* __restrict__ gp,
                                                               unsigned long long* __restrict__ chunk_sum,
                                                               const uint32_t* __restrict__ gate)
{
    __shared__ unsigned long long s_wave[16];
    if (gate && *gate == 0) return;
    const uint32_t bins = BRICKS ? gp->bricks : gp->cells;
    const uint32_t nb   = (bins + kScanChunk - 1) / kScanChunk;
    for (uint32_t b = blockIdx.x; b < nb; b += gridDim.x)
    {
        uint32_t v[8];
        scan_load(count, (size_t)b * kScanChunk + (size_t)threadIdx.x * 8, bins, v);
        unsigned long long sum = 0, total;
#pragma unroll
        for (int k = 0; k < 8; ++k) sum += (unsigned long long)v[k] | (BRICKS && v[k] ? 1ull << 32 : 0ull);
        block_exclusive_scan_1024(sum, s_wave, &total);
        if (threadIdx.x == 0) chunk_sum[b] = total;
    }
}

// start[b]: first point of bin b.  BRICKS also: slot[b] (kNoBrick: the brick is empty), slot_brick[slot], the number of
// slots, and the end of the last cell (cell_start holds one word more than the cells of the bricks).
// not BRICKS also: start[bins] = number of points.
template <bool BRICKS>
__global__ __launch_bounds__(1024) void knn_scan_apply_kernel(const uint32_t* __restrict__ count,
                                                              const KnnGrid* __restrict__ gp,
                                                              const unsigned long long* __restrict__ chunk_sum,
                                                              uint32_t* __restrict__ start, uint32_t* __restrict__ slot,
                                                              uint32_t* __restrict__ slot_brick,
                                                              uint32_t* __restrict__ num_slots,
                                                              uint32_t* __restrict__ cell_start,
                                                              const uint32_t* __restrict__ gate)
{
    __shared__ unsigned long long s_wave[16];
    if (gate && *gate == 0) return;
    const uint32_t bins = BRICKS ? gp->bricks : gp->cells;
    const uint32_t nb   = (bins + kScanChunk - 1) / kScanChunk;
    const unsigned long long mine = threadIdx.x < nb ? chunk_sum[threadIdx.x] : 0ull;  // nb <= kScanChunks
    for (uint32_t b = blockIdx.x; b < nb; b += gridDim.x)
    {
        const size_t t0 = (size_t)b * kScanChunk + (size_t)threadIdx.x * 8;
        uint32_t v[8];
        scan_load(count, t0, bins, v);
        unsigned long long before, sum = 0, total;
        block_exclusive_scan_1024(threadIdx.x < b ? mine : 0ull, s_wave, &before);
#pragma unroll
        for (int k = 0; k < 8; ++k) sum += (unsigned long long)v[k] | (BRICKS && v[k] ? 1ull << 32 : 0ull);
        const unsigned long long run = before + block_exclusive_scan_1024(sum, s_wave, &total);
        uint32_t point = (uint32_t)run, s = (uint32_t)(run >> 32);
        uint32_t o[8], q[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
        {
            o[k] = point;
            q[k] = v[k] ? s : kNoBrick;
            if (BRICKS && v[k]) slot_brick[s++] = (uint32_t)(t0 + k);
            point += v[k];
        }
        if (t0 + 8 <= bins)
        {
            ((uint4*)(start + t0))[0] = make_uint4(o[0], o[1], o[2], o[3]);
            ((uint4*)(start + t0))[1] = make_uint4(o[4], o[5], o[6], o[7]);
            if (BRICKS)
            {
                ((uint4*)(slot + t0))[0] = make_uint4(q[0], q[1], q[2], q[3]);
                ((uint4*)(slot + t0))[1] = make_uint4(q[4], q[5], q[6], q[7]);
            }
        }
        else
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (t0 + k < bins)
                {
                    start[t0 + k] = o[k];
                    if (BRICKS) slot[t0 + k] = q[k];
                }
        if (b == nb - 1 && threadIdx.x == 0)
        {
            const unsigned long long all = before + total;
            if (BRICKS)
            {
                *num_slots                                = (uint32_t)(all >> 32);
                cell_start[(size_t)(all >> 32) << 7] = (uint32_t)all;
            }
            else
                start[bins] = (uint32_t)all;
        }
    }
}

// The points of every brick in the order of its cells, and the first point of every cell: one wavefront per brick that
// holds points, the 128 counters in LDS.  A brick of a surface holds ~160 points: up to 256 stay in registers between
// the count and the scatter, a fuller brick is read twice.
constexpr int kBrickPer = 4;

__global__ __launch_bounds__(kBlock) void knn_brick_sort_kernel(const float4* __restrict__ in,
                                                                const KnnGrid* __restrict__ gp,
                                                                const uint32_t* __restrict__ num_slots,
                                                                const uint32_t* __restrict__ slot_brick,
                                                                const uint32_t* __restrict__ start,
                                                                const uint32_t* __restrict__ count,
                                                                uint32_t* __restrict__ cell_start,
                                                                float4* __restrict__ out)
{
    __shared__ uint32_t s_count[kBlock / 64][kBrickCells];
    uint32_t* cnt       = s_count[threadIdx.x >> 6];
    const int lane      = threadIdx.x & 63;
    const KnnGrid g     = *gp;
    const uint32_t all  = *num_slots;
    // (s is uniform over the wavefront)
    for (uint32_t s = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); s < all; s += gridDim.x * (kBlock / 64))
    {
        const uint32_t b = slot_brick[s], first = start[b], num = count[b];
        wave_lds_sync();
        cnt[lane]      = 0;
        cnt[lane + 64] = 0;
        wave_lds_sync();
        float4 p[kBrickPer];
        uint32_t cell[kBrickPer], rank[kBrickPer];
        for (uint32_t q0 = 0; q0 < num; q0 += 64 * kBrickPer)
        {
#pragma unroll
            for (int k = 0; k < kBrickPer; ++k)
            {
                const uint32_t q = q0 + k * 64 + lane;
                p[k]             = q < num ? in[first + q] : make_float4(0, 0, 0, 0);
            }
#pragma unroll
            for (int k = 0; k < kBrickPer; ++k)
            {
                const int3 c = grid_cell(g, p[k].x, p[k].y, p[k].z);
                cell[k]      = brick_local(c.x, c.y, c.z);
                rank[k]      = q0 + k * 64 + lane < num ? atomicAdd(&cnt[cell[k]], 1u) : 0u;
            }
        }
        wave_lds_sync();
        const uint32_t c0 = cnt[2 * lane], c1 = cnt[2 * lane + 1];
        uint32_t inc = c0 + c1;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1)
        {
            const uint32_t u = (uint32_t)__shfl_up((int)inc, off, 64);
            if (lane >= off) inc += u;
        }
        const uint32_t at = first + inc - c0 - c1;
        ((uint2*)(cell_start + ((size_t)s << 7)))[lane] = make_uint2(at, at + c0);
        wave_lds_sync();
        cnt[2 * lane]     = at;
        cnt[2 * lane + 1] = at + c0;
        wave_lds_sync();
        if (num <= 64 * kBrickPer)
        {
#pragma unroll
            for (int k = 0; k < kBrickPer; ++k)
                if (k * 64 + (uint32_t)lane < num) out[cnt[cell[k]] + rank[k]] = p[k];
        }
        else
            for (uint32_t q = lane; q < num; q += 64)
            {
                const float4 o = in[first + q];
                const int3 c   = grid_cell(g, o.x, o.y, o.z);
                out[atomicAdd(&cnt[brick_local(c.x, c.y, c.z)], 1u)] = o;
            }
    }
}

// ---- search -----------------------------------------------------------------------------------------------------
// A candidate into the ascending list of the K smallest: every place takes the middle one of its left neighbour, the
// candidate and itself.
template <int K>
__device__ __forceinline__ void keep_smallest(float* best, float d2)
{
#pragma unroll
    for (int k = K - 1; k > 0; --k) best[k] = __builtin_amdgcn_fmed3f(best[k - 1], d2, best[k]);
    best[0] = fminf(best[0], d2);
}

__device__ __forceinline__ float distance2(const float4 p, const float4 o)
{
    const float dx = p.x - o.x, dy = p.y - o.y, dz = p.z - o.z;
    return (dx * dx + dy * dy) + dz * dz;
}

// Nothing outside the cube of r shells around cell c is closer than the nearest face of the cube that has cells behind
// it (slightly shrunk: the cell of a point and the faces are computed in fp32).  3e38: the cube is the whole grid.
__device__ __forceinline__ float cube_bound(const KnnGrid& g, const float4 p, int3 c, int r)
{
    float bound = 3.0e38f;
    if (c.x - r > 0) bound = fminf(bound, p.x - (g.min[0] + (float)(c.x - r) * g.cell));
    if (c.y - r > 0) bound = fminf(bound, p.y - (g.min[1] + (float)(c.y - r) * g.cell));
    if (c.z - r > 0) bound = fminf(bound, p.z - (g.min[2] + (float)(c.z - r) * g.cell));
    if (c.x + r < g.dim[0] - 1) bound = fminf(bound, (g.min[0] + (float)(c.x + r + 1) * g.cell) - p.x);
    if (c.y + r < g.dim[1] - 1) bound = fminf(bound, (g.min[1] + (float)(c.y + r + 1) * g.cell) - p.y);
    if (c.z + r < g.dim[2] - 1) bound = fminf(bound, (g.min[2] + (float)(c.z + r + 1) * g.cell) - p.z);
    return fmaxf(bound, 0.f) * 0.999f;
}
__device__ __forceinline__ bool cube_settles(float kth, float bound)
{
    return bound >= 1.0e38f || kth <= bound * bound;
}

// Appends `value` of the lanes with `push` to a list (one atomic per wavefront).  Called by all lanes of a wavefront.
__device__ __forceinline__ void wave_push(bool push, uint32_t value, uint32_t* __restrict__ list, uint32_t* count)
{
    const unsigned long long m = __ballot(push);
    if (!m) return;
    const int lane   = threadIdx.x & 63;
    const int leader = __ffsll((long long)m) - 1;
    uint32_t base    = 0;
    if (lane == leader) base = atomicAdd(count, (uint32_t)__popcll(m));
    base = (uint32_t)__shfl((int)base, leader, 64);
    if (push) list[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = value;
}

// Stage 1: every point, one thread each in the order of the search grid, the cube of 3 x 3 x 3 cells around its own: 9
// rows of cells, each one run of consecutive points, or two where the row crosses into the next brick.  The runs are
// looked up first, all of them at once (two dependent round trips), and kept in LDS; the candidates then come in ONE
// loop over all runs, so that a wavefront takes as many rounds as its fullest cube has candidates and not, row after
// row, as the fullest row.  Points whose n-th neighbour may lie outside the cube go to list.
constexpr int kMaxRuns = 18;
constexpr int kUnroll  = 6;  // candidates of a run per round, their loads in flight together (10 M points on patches, whole
                             // call: 1: 1720 us, 2: 1490, 4: 1300, 6: 1264, 8: 1279)

template <int K>  // K = n + 1 best squared distances are kept (the point itself is one of them)
__global__ __launch_bounds__(kBlock) void knn_search_kernel(KnnView kv, int n, float* __restrict__ out,
                                                            uint32_t* __restrict__ list, uint32_t* list_count)
{
    __shared__ uint2 s_run[kMaxRuns][kBlock];
    const int t     = blockIdx.x * kBlock + threadIdx.x;
    const KnnGrid g = *kv.grid;
    const float4 p  = kv.sorted[t < n ? t : n - 1];
    const int3 c    = grid_cell(g, p.x, p.y, p.z);
    const int x0 = max(c.x - 1, 0), x1 = min(c.x + 1, g.dim[0] - 1);
    const bool two = (x0 >> kBrickX) != (x1 >> kBrickX);
    int runs       = 0;
    for (int part = 0; part < 2; ++part)
    {
        if (part == 1 && !__ballot(two)) break;
        const int xa = part == 0 ? x0 : (x1 >> kBrickX) << kBrickX;
        const int xb = part == 0 && two ? (x0 | 7) : x1;
        uint32_t slot[9], first[9], end[9];
#pragma unroll
        for (int q = 0; q < 9; ++q)
        {
            const int cy = c.y + q % 3 - 1, cz = c.z + q / 3 - 1;
            const bool ok = (unsigned)cy < (unsigned)g.dim[1] && (unsigned)cz < (unsigned)g.dim[2] && (part == 0 || two);
            slot[q]       = ok ? kv.slot[brick_row(g, cy, cz) + (uint32_t)(xa >> kBrickX)] : kNoBrick;
        }
#pragma unroll
        for (int q = 0; q < 9; ++q)
        {
            first[q] = end[q] = 0;
            if (slot[q] != kNoBrick) brick_range(kv, slot[q], xa, xb, c.y + q % 3 - 1, c.z + q / 3 - 1, &first[q], &end[q]);
        }
#pragma unroll
        for (int q = 0; q < 9; ++q)
            if (end[q] > first[q]) s_run[runs++][threadIdx.x] = make_uint2(first[q], end[q]);
    }
    float best[K];
#pragma unroll
    for (int k = 0; k < K; ++k) best[k] = 3.0e38f;
    uint32_t q = 0, e = 0;
    int next = 0;
    for (;;)
    {
        if (q >= e)
        {
            if (next == runs) break;
            const uint2 r = s_run[next++][threadIdx.x];
            q             = r.x;
            e             = r.y;
        }
        float4 o[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) o[u] = kv.sorted[min(q + u, e - 1)];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) keep_smallest<K>(best, q + u < e ? distance2(p, o[u]) : 3.0e38f);
        q += kUnroll;
    }
    const bool settled = cube_settles(best[K - 1], cube_bound(g, p, c, 1));
    if (t < n && settled) out[__float_as_uint(p.w)] = sqrtf(best[K - 1]);
    wave_push(t < n && !settled, (uint32_t)t, list, list_count);
}

// K-th smallest of the union of the lanes' ascending lists (destroys them): K rounds of taking the smallest head.
// all != null receives the K smallest.
template <int K>
__device__ __forceinline__ float wave_kth(float* best, float* all = nullptr)
{
    const int lane = threadIdx.x & 63;
    float kth      = 3.0e38f;
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        float m = best[0];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) m = fminf(m, __shfl_xor(m, off, 64));
        kth = m;
        if (all && lane == 0) all[k] = m;
        const unsigned long long holders = __ballot(best[0] == m);
        if (lane == __ffsll((long long)holders) - 1)
        {
#pragma unroll
            for (int j = 0; j + 1 < K; ++j) best[j] = best[j + 1];
            best[K - 1] = 3.0e38f;
        }
    }
    return kth;
}

// Stage 2: the points stage 1 left, cubes of 2 and 3 shells of the same grid, one wavefront per point: the lanes
// share the rows of the cube (a thread per point waits for 25 to 49 rows one after the other, and few points are
// left: 250 us for a list that a wavefront per point works off in 15).  A larger cube is searched from scratch; the
// rest goes to list2.
template <int K>
__global__ __launch_bounds__(kBlock) void knn_shells_kernel(KnnView kv, const uint32_t* __restrict__ list,
                                                            const uint32_t* __restrict__ list_count,
                                                            float* __restrict__ out, uint32_t* __restrict__ list2,
                                                            uint32_t* list2_count)
{
    const uint32_t count = *list_count;
    const KnnGrid g      = *kv.grid;
    const int lane       = threadIdx.x & 63;
    for (uint32_t e = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); e < count; e += gridDim.x * (kBlock / 64))
    {
        const uint32_t t = list[e];
        const float4 p   = kv.sorted[t];
        const int3 c     = grid_cell(g, p.x, p.y, p.z);
        bool left        = true;
        for (int r = 2; r <= 3 && left; ++r)  // (uniform over the wavefront)
        {
            float best[K];
#pragma unroll
            for (int k = 0; k < K; ++k) best[k] = 3.0e38f;
            const int x0 = max(c.x - r, 0), x1 = min(c.x + r, g.dim[0] - 1);
            const int rows = 2 * r + 1;
            for (int q = lane; q < 2 * rows * rows; q += 64)  // (a row lies in two bricks at most)
            {
                const int row = q >> 1, part = (x0 >> kBrickX) + (q & 1);
                const int cy = c.y - r + row % rows, cz = c.z - r + row / rows;
                if ((unsigned)cy >= (unsigned)g.dim[1] || (unsigned)cz >= (unsigned)g.dim[2] || part > x1 >> kBrickX) continue;
                const uint32_t slot = kv.slot[brick_row(g, cy, cz) + (uint32_t)part];
                if (slot == kNoBrick) continue;
                uint32_t i, end;
                brick_range(kv, slot, max(x0, part << kBrickX), min(x1, part << kBrickX | 7), cy, cz, &i, &end);
                for (; i < end; ++i) keep_smallest<K>(best, distance2(p, kv.sorted[i]));
            }
            const float kth = wave_kth<K>(best);
            if (cube_settles(kth, cube_bound(g, p, c, r)))
            {
                if (lane == 0) out[__float_as_uint(p.w)] = sqrtf(kth);
                left = false;
            }
        }
        if (left && lane == 0) list2[atomicAdd(list2_count, 1u)] = t;
    }
}

// The K-th smallest squared distance of point p on the coarse grid: cubes of 1 to 4 shells, by one wavefront (every
// lane takes its share of the candidates of a row and keeps the K best of them).  False: 4 shells do not settle it.
// Uniform over the wavefront.
template <int K>
__device__ __forceinline__ bool coarse_cubes(const float4 p, const KnnGrid& g, const float4* __restrict__ sorted,
                                             const uint32_t* __restrict__ start, float* kth)
{
    const int lane = threadIdx.x & 63;
    const int3 c   = grid_cell(g, p.x, p.y, p.z);
    for (int r = 1; r <= 4; ++r)
    {
        float best[K];
#pragma unroll
        for (int k = 0; k < K; ++k) best[k] = 3.0e38f;
        const int x0 = max(c.x - r, 0), x1 = min(c.x + r, g.dim[0] - 1);
        for (int cz = max(c.z - r, 0); cz <= min(c.z + r, g.dim[2] - 1); ++cz)
            for (int cy = max(c.y - r, 0); cy <= min(c.y + r, g.dim[1] - 1); ++cy)
            {
                const uint32_t row = grid_index(g, 0, cy, cz), e = start[row + x1 + 1];
                for (uint32_t q = start[row + x0] + lane; q < e; q += 64) keep_smallest<K>(best, distance2(p, sorted[q]));
            }
        *kth = wave_kth<K>(best);
        if (cube_settles(*kth, cube_bound(g, p, c, r))) return true;
    }
    return false;
}

// Stage 3: what is left (points in sparse parts of the cloud), on the coarse grid over all points, at most 4 shells,
// one wavefront per point; the rest goes to list3.
template <int K>
__global__ __launch_bounds__(kBlock) void knn_coarse_kernel(const float4* __restrict__ points,
                                                            const uint32_t* __restrict__ list,
                                                            const uint32_t* __restrict__ list_count,
                                                            const float4* __restrict__ sorted0,
                                                            const KnnGrid* __restrict__ gp0,
                                                            const uint32_t* __restrict__ start0, float* __restrict__ out,
                                                            uint32_t* __restrict__ list3, uint32_t* list3_count)
{
    const uint32_t count = *list_count;
    const KnnGrid g      = *gp0;
    const int lane       = threadIdx.x & 63;
    for (uint32_t e = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); e < count; e += gridDim.x * (kBlock / 64))
    {
        const uint32_t t = list[e];
        const float4 p   = points[t];
        float kth;
        if (coarse_cubes<K>(p, g, sorted0, start0, &kth))
        {
            if (lane == 0) out[__float_as_uint(p.w)] = sqrtf(kth);
        }
        else if (lane == 0)
            list3[atomicAdd(list3_count, 1u)] = t;
    }
}

// Stage 4: stray points far from everything (no cube of a few shells of either grid settles them): one workgroup goes
// through all points for one of them, or for kBruteStrays together where there are more strays than workgroups.  (A
// wavefront per stray, 1 M points of a Gaussian cloud: 1.5 ms; a workgroup of 16: 0.25 ms - there are fewer strays
// than the GPU has wavefronts.)  With thousands of strays the points come from the last cache over and over, 5 TB/s
// of them, so strays share a pass; of the thousands of points a thread sees few get into its lists, so a round of
// kBruteRound points is looked at as a whole before any of it goes in.  6 M points of a Gaussian cloud, rank 4 / 8
// (some 1500 / 4000 strays): one stray per pass 29.8 / 77.5 ms, four 6.2 / 14.3.
constexpr int kBruteBlock  = 1024;
constexpr int kBruteStrays = 4;
constexpr int kBruteRound  = 4;

template <int K, int S>
__device__ __forceinline__ void brute_pass(const float4* __restrict__ points, int n, const uint32_t* __restrict__ list,
                                           uint32_t first, uint32_t count, float (*s_best)[kBruteBlock / 64][K],
                                           float* __restrict__ out)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float4 p[S];
    float best[S][K];
#pragma unroll
    for (int s = 0; s < S; ++s)
    {
        p[s] = points[list[first + s < count ? first + s : count - 1]];
#pragma unroll
        for (int k = 0; k < K; ++k) best[s][k] = 3.0e38f;
    }
    for (size_t q0 = threadIdx.x; q0 < (size_t)n; q0 += kBruteRound * kBruteBlock)
    {
        float4 o[kBruteRound];
#pragma unroll
        for (int u = 0; u < kBruteRound; ++u)
        {
            const size_t q = q0 + u * kBruteBlock;
            o[u]           = points[q < (size_t)n ? q : (size_t)n - 1];
        }
#pragma unroll
        for (int s = 0; s < S; ++s)
        {
            float d2[kBruteRound], nearest = 3.0e38f;
#pragma unroll
            for (int u = 0; u < kBruteRound; ++u)
            {
                d2[u]   = q0 + u * kBruteBlock < (size_t)n ? distance2(p[s], o[u]) : 3.0e38f;
                nearest = fminf(nearest, d2[u]);
            }
            if (nearest < best[s][K - 1])
            {
#pragma unroll
                for (int u = 0; u < kBruteRound; ++u) keep_smallest<K>(best[s], d2[u]);
            }
        }
    }
#pragma unroll
    for (int s = 0; s < S; ++s) wave_kth<K>(best[s], s_best[s][wave]);
    __syncthreads();
    if (wave < S && first + wave < count)  // the wavefronts' lists of one stray, one per lane
    {
        float all[K];
#pragma unroll
        for (int k = 0; k < K; ++k) all[k] = lane < kBruteBlock / 64 ? s_best[wave][lane][k] : 3.0e38f;
        const float kth = wave_kth<K>(all);
        if (lane == 0) out[__float_as_uint(points[list[first + wave]].w)] = sqrtf(kth);
    }
    __syncthreads();  // s_best has been read
}

template <int K>
__global__ __launch_bounds__(kBruteBlock) void knn_brute_kernel(const float4* __restrict__ points, int n,
                                                                const uint32_t* __restrict__ list,
                                                                const uint32_t* __restrict__ list_count,
                                                                float* __restrict__ out)
{
    __shared__ float s_best[kBruteStrays][kBruteBlock / 64][K];
    static_assert(kBruteStrays <= kBruteBlock / 64, "one wavefront per stray at the end");
    const uint32_t count = *list_count;  // (all branches on it are uniform over the grid)
    if (count <= gridDim.x)
    {
        if (blockIdx.x < count) brute_pass<K, 1>(points, n, list, blockIdx.x, count, s_best, out);
    }
    else
        for (uint32_t e = blockIdx.x * kBruteStrays; e < count; e += gridDim.x * kBruteStrays)
            brute_pass<K, kBruteStrays>(points, n, list, e, count, s_best, out);
}

// The neighbour distance of `samples` points evenly spaced in the order of the coarse grid, one wavefront per point
// (the lanes share the candidates, every lane keeps the K best of its share).  out[s] = distance of sample s, 3e38
// for a sample that 4 shells do not settle (a stray point: it shall not size the grid).  All branches on r, the bound
// and the result are uniform over the wavefront.
template <int K>
__global__ __launch_bounds__(kBlock) void knn_sample_kernel(const float4* __restrict__ sorted, int n,
                                                            const KnnGrid* __restrict__ gp,
                                                            const uint32_t* __restrict__ offset, float* __restrict__ out,
                                                            int samples)
{
    const int slot = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (slot >= samples) return;
    const int t     = (int)((long long)slot * n / samples);
    float kth;
    const bool settled = coarse_cubes<K>(sorted[t], *gp, sorted, offset, &kth);
    if (lane == 0) out[slot] = settled ? sqrtf(kth) : 3.0e38f;
}

// ---- sizing the grids -------------------------------------------------------------------------------------------
constexpr int kKnnSamples   = 1024;
constexpr int kKnnMaxDim    = 2048;
constexpr int kKnnCoarseDim = 160;
static_assert(kKnnCoarseDim * kKnnCoarseDim * kKnnCoarseDim <= kScanChunk * kScanChunks, "chunks of the coarse grid");
static_assert(kKnnMaxBricks <= (size_t)kScanChunk * kScanChunks, "chunks of the search grid");

// A = 1 or 3 arrays of kKnnSamples floats in LDS, each sorted ascending by a workgroup of 1024 threads (bitonic; the
// arrays share the barriers)
template <int A>
__device__ __forceinline__ void sort_samples(float (*s)[kKnnSamples])
{
    for (int k = 2; k <= kKnnSamples; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1)
        {
            for (int w = threadIdx.x; w < A * (kKnnSamples / 2); w += 1024)
            {
                float* a    = s[w / (kKnnSamples / 2)];
                const int h = w & (kKnnSamples / 2 - 1);
                const int i = ((h & ~(j - 1)) << 1) | (h & (j - 1)), o = i | j;
                const float u = a[i], v = a[o];
                if ((u > v) == ((i & k) == 0))
                {
                    a[i] = v;
                    a[o] = u;
                }
            }
            __syncthreads();
        }
}

// Coarse grid.  Its box is not the bounding box of the cloud (one far outlier would stretch that until all other points
// share a cell) but, per axis, the 1st to 99th percentile of 1024 points taken at equal steps through the array,
// widened by 5 % of that range on either side and cut to the caller's box; the points outside it go to the boundary
// cells, which keeps the search exact (a cube of cells then stands for a region open to the outside).  Cells for ~8
// points each if the cloud filled the box, at most kKnnCoarseDim per axis.  One workgroup.
__global__ __launch_bounds__(1024) void knn_first_grid_kernel(const float4* __restrict__ position, int n, KnnGrid box,
                                                              KnnGrid* __restrict__ dst)
{
    __shared__ float s[3][kKnnSamples];
    const int samples = n < kKnnSamples ? n : kKnnSamples;
    {
        static_assert(kKnnSamples == 1024, "one sample per thread");
        const int i = threadIdx.x;
        float4 p    = make_float4(3.0e38f, 3.0e38f, 3.0e38f, 0.f);
        if (i < samples) p = position[(size_t)((long long)i * n / samples)];
        s[0][i] = p.x;
        s[1][i] = p.y;
        s[2][i] = p.z;
    }
    __syncthreads();
    sort_samples<3>(s);
    if (threadIdx.x != 0) return;
    KnnGrid g;
    for (int k = 0; k < 3; ++k)
    {
        const float a = s[k][samples / 100], b = s[k][samples - 1 - samples / 100];
        const float box_hi = box.min[k] + box.ext[k];
        float lo = fmaxf(a - 0.05f * (b - a), box.min[k]), hi = fminf(b + 0.05f * (b - a), box_hi);
        if (!(hi >= lo))  // not a number among the samples
        {
            lo = box.min[k];
            hi = box_hi;
        }
        g.min[k] = lo;
        g.ext[k] = hi - lo;
    }
    const float longest = fmaxf(g.ext[0], fmaxf(g.ext[1], g.ext[2]));
    float volume        = 1.f;  // thin axes count as a millionth of the longest one
    for (int k = 0; k < 3; ++k) volume *= g.ext[k] > 1e-6f * longest ? g.ext[k] : (longest > 0.f ? 1e-6f * longest : 1.f);
    float cell = cbrtf(volume * 8.0f / (float)n);
    if (!(cell > longest / kKnnCoarseDim)) cell = longest / kKnnCoarseDim;
    if (!(cell > 0.f)) cell = 1.f;  // all samples coincide
    g.cell     = cell;
    g.inv_cell = 1.0f / cell;
    g.cells    = 1;
    for (int k = 0; k < 3; ++k)
    {
        int d    = (int)(g.ext[k] / cell) + 1;
        g.dim[k] = d < 1 ? 1 : (d > kKnnCoarseDim ? kKnnCoarseDim : d);
        g.cells *= (uint32_t)g.dim[k];
    }
    g.bricks_x = g.bricks_y = 0;
    g.bricks                = 0;
    *dst                    = g;
}

// Search grid: cells of `factor` times the median sampled neighbour distance, never coarser than the coarse grid, at
// most kKnnMaxDim cells per axis and `budget` bricks in all, over the same box.  One workgroup.  Also clears the list
// counters of the search.
__global__ __launch_bounds__(1024) void knn_refine_grid_kernel(const float* __restrict__ sample, int samples, float factor,
                                                               const KnnGrid* __restrict__ first,
                                                               KnnGrid* __restrict__ gp, uint32_t budget,
                                                               uint32_t* __restrict__ list_counts)
{
    __shared__ float s[1][kKnnSamples];
    s[0][threadIdx.x] = (int)threadIdx.x < samples ? sample[threadIdx.x] : 3.0e38f;
    if (threadIdx.x < 3) list_counts[threadIdx.x] = 0;
    __syncthreads();
    sort_samples<1>(s);
    if (threadIdx.x != 0) return;
    KnnGrid g           = *first;
    const float median  = s[0][samples / 2];
    const float longest = fmaxf(g.ext[0], fmaxf(g.ext[1], g.ext[2]));
    float cell = factor * median;
    if (!(cell < g.cell)) cell = g.cell;  // also NaN / the 3e38 of a cloud with fewer points than neighbours asked for
    if (!(cell > longest / (float)(kKnnMaxDim - 1))) cell = longest / (float)(kKnnMaxDim - 1);
    if (!(cell > 0.f)) cell = g.cell;
    for (;;)
    {
        uint32_t b[3];
        for (int k = 0; k < 3; ++k)
        {
            int d    = (int)(g.ext[k] / cell) + 1;
            g.dim[k] = d < 1 ? 1 : (d > kKnnMaxDim ? kKnnMaxDim : d);
            b[k]     = k == 0 ? ((uint32_t)g.dim[k] + 7) >> kBrickX : ((uint32_t)g.dim[k] + 3) >> kBrickY;
        }
        const unsigned long long bricks = (unsigned long long)b[0] * b[1] * b[2];
        if (bricks <= budget)
        {
            g.bricks_x = (int)b[0];
            g.bricks_y = (int)b[1];
            g.bricks   = (uint32_t)bricks;
            break;
        }
        cell *= 1.1f;
    }
    g.cell     = cell;
    g.inv_cell = 1.0f / cell;
    *gp        = g;
}

// One frame of it: the squared distance of the point, if the frame sees it and it is smaller.
__device__ __forceinline__ void nearest_camera(const ViewConst& vc, V3 pos, float* best)
{
    const V3 r = quat_rotate(vc.qx, vc.qy, vc.qz, vc.qw, pos);
    const V3 v = {r.x + vc.tx, r.y + vc.ty, r.z + vc.tz};
    const float d = (v.x * v.x + v.y * v.y) + v.z * v.z;
    if (!(v.z > 0.f) || !(d < *best)) return;
    const V2 np   = {v.x / v.z, v.y / v.z};
    const V2 dp   = distort<false>(np, vc.d, 3.0e38f, nullptr, nullptr);
    const V2 ip   = k_apply(vc.k, dp);
    const bool in = ip.x >= 0.f && ip.y >= 0.f && ip.x < (float)vc.w && ip.y < (float)vc.h;
    if (in) *best = d;
}

// SceneData::PointDistanceToCamera (SceneData.cpp:645-669): distance from every point to the nearest camera that sees
// it (in front of the camera, projected inside the image with the frame's pinhole + distortion model), 10258.4 (the
// root of the reference's start value 105235545) where no frame does.  The distance is taken in camera space
// (|V p| = |p - c| for the camera centre c).  The frames are read through uniform loads.
__global__ __launch_bounds__(kBlock) void camera_distance_kernel(const float4* __restrict__ position, int n,
                                                                 const ViewConst* __restrict__ views, int num_frames,
                                                                 float* __restrict__ out)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float4 P = nt_load4(position + i);
    const V3 pos   = {P.x, P.y, P.z};
    float best     = 105235545.f;
    for (int f = 0; f < num_frames; ++f) nearest_camera(views[f], pos, &best);
    out[i] = sqrtf(best);
}

// The same for points in the order of the search grid: a wavefront's points lie close together, so most frames are
// ruled out for all of them at once.  Per 64 frames, every lane takes one: a bound below the distance of its camera
// to any point of the wavefront's bounding sphere, or none if the whole sphere lies behind the camera.  The frames
// then come nearest first, until the next bound is above what every lane has found.  The minimum over the frames that
// see a point does not depend on their order, and the bound leaves 1e-5 of the coordinates for rounding. 3 M points
// of a sphere on a plane, 100 frames: 708 -> 307 us (the corners of the plane are in few images, and a point no frame
// sees takes all of them).
__global__ __launch_bounds__(kBlock) void camera_distance_sorted_kernel(const float4* __restrict__ sorted, int n,
                                                                        const ViewConst* __restrict__ views, int num_frames,
                                                                        float* __restrict__ out)
{
    const int t    = blockIdx.x * kBlock + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const float4 P = sorted[t < n ? t : n - 1];
    const V3 pos   = {P.x, P.y, P.z};
    const float lo[3] = {wave_min(P.x), wave_min(P.y), wave_min(P.z)}, hi[3] = {wave_max(P.x), wave_max(P.y), wave_max(P.z)};
    const V3 c     = {0.5f * (lo[0] + hi[0]), 0.5f * (lo[1] + hi[1]), 0.5f * (lo[2] + hi[2])};
    const V3 half  = {hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]};
    const float radius = 0.5f * sqrtf(dot3(half, half));
    float best     = 105235545.f;
    for (int f0 = 0; f0 < num_frames; f0 += 64)
    {
        const float never = __builtin_inff();
        float bound       = never;
        if (f0 + lane < num_frames)
        {
            const ViewConst& vc = views[f0 + lane];
            const V3 r = quat_rotate(vc.qx, vc.qy, vc.qz, vc.qw, c);
            const V3 v = {r.x + vc.tx, r.y + vc.ty, r.z + vc.tz};
            const float size  = fabsf(c.x) + fabsf(c.y) + fabsf(c.z) + radius + fabsf(vc.tx) + fabsf(vc.ty) + fabsf(vc.tz);
            const float slack = radius * 1.0001f + 1.0e-5f * size;
            const float reach = sqrtf(dot3(v, v)) - slack;
            if (!(v.z + slack <= 0.f)) bound = reach > 0.f ? reach * reach * 0.9999f : 0.f;
        }
        for (;;)
        {
            const float next = wave_min(bound);
            if (next == never || next >= wave_max(best)) break;  // (wavefront-uniform)
            const int f = __ffsll((long long)__ballot(bound == next)) - 1;
            nearest_camera(views[f0 + f], pos, &best);
            if (lane == f) bound = never;
        }
    }
    if (t < n) out[__float_as_uint(P.w)] = sqrtf(best);
}

// SceneData::RemoveClosePoints (SceneData.cpp:598-642) walks the points in order and erases point i when a point it
// has kept before lies within radius[i] of it: state[i] = kept unless a kept j < i is that close.  Here the points
// are decided in rounds: a point whose earlier neighbours are all decided is decided; states only ever go from
// undecided to kept / erased, so reading a neighbour's state of this round instead of the last one is as good. One
// thread per point in cell order; count[round] receives the points still undecided after this round, and a round that
// finds count[round - 1] == 0 has nothing to do. The cells a ball can reach are those of the corners of its bounding
// cube: the cell of a coordinate never decreases with it, in fp32 as in real numbers, and a point counts only if
// every |difference of coordinates| is below the radius up to the rounding of four operations, which the widened
// reach covers (1e-4 of the radius; 1e-20 where its square underflows).  The radii of the filter are a hundredth of a
// cell: one row of one or two cells in place of the 27 around the point (3 M points in random order: 730 -> 177 us,
// most of it the states and radii, which are gathered by id). A scene in a unit of its own has radii of many cells
// (the radius grows as the unit, the cells shrink): then the kernel waits for the rows it looks up, one load after
// the other.  One flat loop over candidates, rows and bricks, so that a wavefront takes as many turns as its longest
// lane needs of all of them together and not the longest of every row; where the ball spans a brick in x the rows of
// a layer are one run; candidates and their states come in fours.  Whole call, cells row by row / flat: 1 M points on
// patches, radii of 4 cells 7.0 / 4.8 ms, of a Gaussian cloud 10.7 / 8.2, on a plane and a sphere 15.8 / 14.3; 3 M
// points with radii of a hundredth of a cell 252 / 231 us in this kernel.
constexpr int kStateUndecided = 0, kStateKept = 1, kStateErased = 2;
constexpr int kCloseUnroll    = 4;

__global__ __launch_bounds__(kBlock) void close_points_kernel(KnnView kv, int n, const float* __restrict__ radius,
                                                              int32_t* state, uint32_t* round_count, int round)
{
    if (round > 0 && *(volatile uint32_t*)(round_count + round - 1) == 0) return;
    const int t = blockIdx.x * kBlock + threadIdx.x;
    bool pending = false;
    if (t < n)
    {
        const KnnGrid g  = *kv.grid;
        const float4 p   = kv.sorted[t];
        const uint32_t i = __float_as_uint(p.w);
        if (__atomic_load_n(&state[i], __ATOMIC_RELAXED) == kStateUndecided)
        {
            const float rad = radius[i];
            const float r2  = rad * rad;
            const float reach = fabsf(rad) * 1.0001f + 1.0e-20f;
            const int3 lo   = grid_cell(g, p.x - reach, p.y - reach, p.z - reach);
            const int3 hi   = grid_cell(g, p.x + reach, p.y + reach, p.z + reach);
            int result = kStateKept;
            const int3 b0 = {lo.x >> kBrickX, lo.y >> kBrickY, lo.z >> kBrickZ};
            const int3 b1 = {hi.x >> kBrickX, hi.y >> kBrickY, hi.z >> kBrickZ};
            int3 b        = {b0.x - 1, b0.y, b0.z};  // (no brick yet)
            int xa = 0, xb = 0, ya = 0, yb = 0, zb = -1, cy = 0, cz = 0;
            uint32_t slot = kNoBrick, q = 0, e = 0;
            for (;;)
            {
                if (q < e)
                {
                    float4 o[kCloseUnroll];
#pragma unroll
                    for (int u = 0; u < kCloseUnroll; ++u) o[u] = kv.sorted[min(q + u, e - 1)];
                    // (the states of all candidates that count are requested before the first is looked at; the state
                    // of the point itself, which is undecided and stands in for the others, is not looked at)
                    bool near[kCloseUnroll], any = false;
#pragma unroll
                    for (int u = 0; u < kCloseUnroll; ++u)
                    {
                        near[u] = q + u < e && __float_as_uint(o[u].w) < i && distance2(p, o[u]) < r2;
                        any |= near[u];
                    }
                    if (any)
                    {
                        int32_t sj[kCloseUnroll];
#pragma unroll
                        for (int u = 0; u < kCloseUnroll; ++u)
                            sj[u] = __atomic_load_n(&state[near[u] ? __float_as_uint(o[u].w) : i], __ATOMIC_RELAXED);
#pragma unroll
                        for (int u = 0; u < kCloseUnroll; ++u)
                        {
                            if (near[u] && sj[u] == kStateKept) result = kStateErased;
                            if (near[u] && sj[u] == kStateUndecided && result != kStateErased) result = kStateUndecided;
                        }
                    }
                    if (result == kStateErased) break;
                    q += kCloseUnroll;
                }
                else if (cz <= zb)  // the next row or layer of the brick
                {
                    const int ye        = xb - xa == 7 ? yb : cy;
                    const uint32_t* row = kv.cell_start + ((size_t)slot << 7);
                    q                   = row[brick_local(xa, cy, cz)];
                    e                   = row[brick_local(xb, ye, cz) + 1];
                    cy                  = ye + 1;
                    if (cy > yb)
                    {
                        cy = ya;
                        ++cz;
                    }
                }
                else  // the next brick of the box
                {
                    if (++b.x > b1.x)
                    {
                        b.x = b0.x;
                        if (++b.y > b1.y)
                        {
                            b.y = b0.y;
                            if (++b.z > b1.z) break;
                        }
                    }
                    slot = kv.slot[brick_row(g, b.y << kBrickY, b.z << kBrickZ) + (uint32_t)b.x];
                    xa   = max(lo.x, b.x << kBrickX);
                    xb   = min(hi.x, b.x << kBrickX | 7);
                    ya   = max(lo.y, b.y << kBrickY);
                    yb   = min(hi.y, b.y << kBrickY | 3);
                    cy   = ya;
                    cz   = max(lo.z, b.z << kBrickZ);
                    zb   = slot == kNoBrick ? -1 : min(hi.z, b.z << kBrickZ | 3);
                }
            }
            if (result != kStateUndecided) __atomic_store_n(&state[i], result, __ATOMIC_RELAXED);
            pending = result == kStateUndecided;
        }
    }
    const unsigned long long m = __ballot(pending);
    if (m && (threadIdx.x & 63) == (__ffsll((long long)m) - 1)) atomicAdd(round_count + round, (uint32_t)__popcll(m));
}

// Morton code of every point: 21 bits per axis of the position inside the bounding box, x in the lowest bit.
__device__ __forceinline__ unsigned long long spread21(unsigned long long v)
{
    v &= 0x1FFFFFull;
    v = (v | v << 32) & 0x1F00000000FFFFull;
    v = (v | v << 16) & 0x1F0000FF0000FFull;
    v = (v | v << 8) & 0x100F00F00F00F00Full;
    v = (v | v << 4) & 0x10C30C30C30C30C3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}

// key (may be null): the upper 32 bits of the code, as a signed number in the same order.
__global__ __launch_bounds__(kBlock) void morton_kernel(const float4* __restrict__ position, int n, float min_x,
                                                        float min_y, float min_z, float scale_x, float scale_y,
                                                        float scale_z, unsigned long long* __restrict__ code,
                                                        int32_t* __restrict__ key)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float4 p = nt_load4(position + i);
    const float m  = 2097151.f;  // 2^21 - 1
    const float fx = fminf(fmaxf((p.x - min_x) * scale_x, 0.f), m);
    const float fy = fminf(fmaxf((p.y - min_y) * scale_y, 0.f), m);
    const float fz = fminf(fmaxf((p.z - min_z) * scale_z, 0.f), m);
    const unsigned long long c = spread21((unsigned long long)fx) | spread21((unsigned long long)fy) << 1 |
                                 spread21((unsigned long long)fz) << 2;
    code[i] = c;
    if (key) key[i] = (int32_t)((uint32_t)(c >> 31) ^ 0x80000000u);
}

// `order` sorts the points stably by `key`, the upper half of their codes (sorted_key: the keys in that order); the
// points of equal keys are put in the order of their whole codes, equal codes staying as they are.  The first point
// of a run of equal keys does it, by insertion: a run is two or three points where the cloud fills its bounding box.
// A run of more than kTieRun points is left alone and *too_long set: the caller then sorts by whole codes. 10 M
// points, sort and ties: by whole codes (11 passes) 974 us, by keys (6 shorter ones) 539 us in a volume, 688 on
// patches, 796 on a plane and a sphere (more ties); 1 M: 238 against 216 to 226; 300 k: 159 against 157, and the flag
// is still to be read.
constexpr int kTieRun = 32;

__global__ __launch_bounds__(kBlock) void morton_ties_kernel(const int32_t* __restrict__ sorted_key, long long* __restrict__ order,
                                                             const unsigned long long* __restrict__ code, int n,
                                                             int32_t* too_long)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n - 1) return;
    const int32_t key = sorted_key[i];
    if (key != sorted_key[i + 1] || (i > 0 && key == sorted_key[i - 1])) return;
    int end = i + 2;
    while (end < n && end - i <= kTieRun && sorted_key[end] == key) ++end;
    if (end - i > kTieRun)
    {
        *too_long = 1;
        return;
    }
    for (int a = i + 1; a < end; ++a)
    {
        const long long id         = order[a];
        const unsigned long long c = code[id];
        int to                     = a;
        while (to > i && code[order[to - 1]] > c)
        {
            order[to] = order[to - 1];
            --to;
        }
        order[to] = id;
    }
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
int knn_sample_stride(int n) { return n >= (1 << 17) ? 16 : 1; }
int knn_num_samples(int n) { return n < kKnnSamples ? n : kKnnSamples; }
size_t knn_chunk_words() { return 2 * (size_t)kScanChunks; }

void launch_knn_first_grid(const float4* position, int n, const KnnGrid& box, KnnGrid* dst, hipStream_t st)
{
    hipLaunchKernelGGL(knn_first_grid_kernel, dim3(1), dim3(1024), 0, st, position, n, box, dst);
}

// The cells of the search grid as a multiple of the median distance d_R to the R-th neighbour.  Smaller cells mean
// fewer candidates (their number goes with the square of the cell on a surface, with the cube in a volume) and more
// points that the cube of 27 cells does not settle.  1.5 measured best over surfaces and volumes (search of 10 M
// points on 1000 patches, 3 M in a volume, whole call: 2.0: 1365, 786 us; 1.5: 1264, 574; 1.2: 1283, 1015).  Where
// the samples are taken in every s-th point, their nearest neighbour there stands in for the s-th in the cloud, and
// d_R = d_s (R / s)^(1 / D) for a cloud of dimension D.  D = 2.5 is 32 % above a surface's value at R = 1, s = 16 and
// 17 % below a volume's, and cells too small by that much leave a seventh of a volume's points unsettled; the
// distance to the nearest neighbour also spreads more about its median than that to the 8th.  R + 1.25 in the place
// of R takes care of both where it matters and costs surfaces nothing (6 M points in a volume, rank 1 / 2 / 4 / 8:
// with R 2.03, 1.87, 1.35, 1.30 ms, with R + 1.25 1.05, 1.06, 1.13, 1.36; 10 M points on patches 2.07 and 2.08).
void launch_knn_refine_grid(const float* sample, int samples, int rank, int stride, const KnnGrid* first, KnnGrid* g,
                            uint32_t budget, uint32_t* list_counts, hipStream_t st)
{
    const float factor = 1.5f * (stride > 1 ? powf(((float)rank + 1.25f) / (float)stride, 0.4f) : 1.0f);
    hipLaunchKernelGGL(knn_refine_grid_kernel, dim3(1), dim3(1024), 0, st, sample, samples, factor, first, g, budget,
                       list_counts);
}

static int bin_blocks(int n) { return (int)(((size_t)n + kBlock * kBinPer - 1) / (kBlock * kBinPer)); }

// every stride-th point (n of them) in the cell order of the coarse grid
void launch_knn_coarse(const float4* position, int n, int stride, const KnnGrid* g, uint32_t* count, uint32_t* start,
                       uint32_t* rank, unsigned long long* chunk_sum, float4* sorted, const uint32_t* gate, hipStream_t st)
{
    hipLaunchKernelGGL(knn_clear_kernel<false>, dim3(1024), dim3(kBlock), 0, st, count, g, gate);
    hipLaunchKernelGGL(knn_count_kernel<false>, dim3(bin_blocks(n)), dim3(kBlock), 0, st, position, n, stride, g, count, rank, gate);
    hipLaunchKernelGGL(knn_scan_reduce_kernel<false>, dim3(512), dim3(1024), 0, st, count, g, chunk_sum, gate);
    hipLaunchKernelGGL(knn_scan_apply_kernel<false>, dim3(512), dim3(1024), 0, st, count, g, chunk_sum, start, nullptr, nullptr,
                       nullptr, nullptr, gate);
    hipLaunchKernelGGL(knn_scatter_kernel<false>, dim3(bin_blocks(n)), dim3(kBlock), 0, st, position, n, stride, g, start, rank,
                       sorted, gate);
}

// the points in the order of the search grid's bricks and cells
void launch_knn_bricks(const float4* position, int n, const KnnBricks& b, hipStream_t st)
{
    const int chunks = (int)((b.max_bricks + kScanChunk - 1) / kScanChunk);
    hipLaunchKernelGGL(knn_clear_kernel<true>, dim3(1024), dim3(kBlock), 0, st, b.count, b.grid, nullptr);
    hipLaunchKernelGGL(knn_count_kernel<true>, dim3(bin_blocks(n)), dim3(kBlock), 0, st, position, n, 1, b.grid, b.count, b.rank,
                       nullptr);
    hipLaunchKernelGGL(knn_scan_reduce_kernel<true>, dim3(chunks), dim3(1024), 0, st, b.count, b.grid, b.chunk_sum, nullptr);
    hipLaunchKernelGGL(knn_scan_apply_kernel<true>, dim3(chunks), dim3(1024), 0, st, b.count, b.grid, b.chunk_sum, b.start, b.slot,
                       b.slot_brick, b.num_slots, b.cell_start, nullptr);
    hipLaunchKernelGGL(knn_scatter_kernel<true>, dim3(bin_blocks(n)), dim3(kBlock), 0, st, position, n, 1, b.grid, b.start, b.rank,
                       b.scratch, nullptr);
    // (as many wavefronts as there can be bricks with points, at most 2 per wave slot of the GPU)
    const size_t slots = (size_t)n < b.max_bricks ? (size_t)n : b.max_bricks;
    const size_t want  = (slots + kBlock / 64 - 1) / (kBlock / 64);
    hipLaunchKernelGGL(knn_brick_sort_kernel, dim3((int)(want < 4096 ? want : 4096)), dim3(kBlock), 0, st, b.scratch, b.grid,
                       b.num_slots, b.slot_brick, b.start, b.count, b.cell_start, b.sorted);
}

#define ADOP_KNN_RANKS                                                                                 \
    ADOP_KNN_CASE(1) ADOP_KNN_CASE(2) ADOP_KNN_CASE(3) ADOP_KNN_CASE(4) ADOP_KNN_CASE(5) ADOP_KNN_CASE(6) \
    ADOP_KNN_CASE(7) ADOP_KNN_CASE(8)

bool launch_knn_sample(int rank, const float4* sorted, int n, const KnnGrid* g, const uint32_t* offset, float* out,
                       int samples, hipStream_t st)
{
    const dim3 block(kBlock), grid((samples + kBlock / 64 - 1) / (kBlock / 64));
#define ADOP_KNN_CASE(R) \
    case R: hipLaunchKernelGGL(knn_sample_kernel<R + 1>, grid, block, 0, st, sorted, n, g, offset, out, samples); return true;
    switch (rank)
    {
        ADOP_KNN_RANKS
    }
#undef ADOP_KNN_CASE
    return false;
}

// The four stages of the search: the cube of 27 cells (all points), 2 and 3 shells, the coarse grid over all points
// (built only if something is left), all points (strays).
bool launch_knn_search(int rank, const float4* position, int n, const KnnSearchArg& a, float* out, hipStream_t st)
{
    const dim3 block(kBlock), grid((n + kBlock - 1) / kBlock), grid2(2048), grid3(512);
#define ADOP_KNN_CASE(R)                                                                                                \
    case R:                                                                                                             \
        hipLaunchKernelGGL(knn_search_kernel<R + 1>, grid, block, 0, st, a.view, n, out, a.list, a.counts);              \
        hipLaunchKernelGGL(knn_shells_kernel<R + 1>, grid2, block, 0, st, a.view, a.list, a.counts, out, a.list2,        \
                           a.counts + 1);                                                                               \
        launch_knn_coarse(position, n, 1, a.grid0, a.count0, a.start0, a.rank, a.chunk_sum, a.sorted0, a.counts + 1, st); \
        hipLaunchKernelGGL(knn_coarse_kernel<R + 1>, grid2, block, 0, st, a.view.sorted, a.list2, a.counts + 1,          \
                           a.sorted0, a.grid0, a.start0, out, a.list, a.counts + 2);                                    \
        hipLaunchKernelGGL(knn_brute_kernel<R + 1>, grid3, dim3(kBruteBlock), 0, st, a.view.sorted, n, a.list, a.counts + 2, out);   \
        return true;
    switch (rank)
    {
        ADOP_KNN_RANKS
    }
#undef ADOP_KNN_CASE
    return false;
}
#undef ADOP_KNN_RANKS

void launch_camera_distance(const float4* position, int n, const ViewConst* views, int num_frames, float* out,
                            hipStream_t st)
{
    hipLaunchKernelGGL(camera_distance_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, position, n, views,
                       num_frames, out);
}

void launch_camera_distance_sorted(const float4* sorted, int n, const ViewConst* views, int num_frames, float* out,
                                   hipStream_t st)
{
    hipLaunchKernelGGL(camera_distance_sorted_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, sorted, n, views,
                       num_frames, out);
}

void launch_close_points(const KnnView& view, int n, const float* radius, int32_t* state, uint32_t* round_count, int round,
                         hipStream_t st)
{
    hipLaunchKernelGGL(close_points_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, view, n, radius, state,
                       round_count, round);
}

void launch_morton(const float4* position, int n, const float* mn, const float* scale, unsigned long long* code, int32_t* key,
                   hipStream_t st)
{
    hipLaunchKernelGGL(morton_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, position, n, mn[0], mn[1],
                       mn[2], scale[0], scale[1], scale[2], code, key);
}

void launch_morton_ties(const int32_t* sorted_key, long long* order, const unsigned long long* code, int n, int32_t* too_long,
                        hipStream_t st)
{
    hipLaunchKernelGGL(morton_ties_kernel, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, sorted_key, order, code, n, too_long);
}

}  // namespace adop
