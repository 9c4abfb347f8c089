// cloud_kernels.h — included by preprocess_kernels.hip alone: moving whole clouds (gfx950): bounding box,
// permutations of the points, radii and order of the 256-point blocks.  The counterpart of the loops of
// SceneData.cpp:101-104 and :441-484, 671-684 that touch every point once; what they compute per point is next to
// nothing, so these kernels are bound by memory: random 64-byte lines where they gather, the bandwidth of a copy
// where they do not.
#pragma once
#include "common.h"
#include "launch.h"

#pragma clang fp contract(off)

namespace adop
{
// ---- bounding box -----------------------------------------------------------------------------------------------
// Smallest and largest x, y, z; a coordinate that is not a number makes both ends of its axis not a number (the
// caller's check of the box then fails).  Two launches: kBoxBlocks partial boxes, then one workgroup over them.
// 10 M points (160 MB): 28 + 11 us, 5.7 TB/s in the first (torch.aminmax over the rows: 77 us).
constexpr int kBoxBlocks = 2048;

struct Box6
{
    float lo[3], hi[3];
};

__device__ __forceinline__ Box6 empty_box()
{
    const float inf = __builtin_inff();
    return Box6{{inf, inf, inf}, {-inf, -inf, -inf}};
}
__device__ __forceinline__ float min_nan(float a, float b) { return a != a ? a : (b != b ? b : fminf(a, b)); }
__device__ __forceinline__ float max_nan(float a, float b) { return a != a ? a : (b != b ? b : fmaxf(a, b)); }

__device__ __forceinline__ void box_of_block(Box6& box, float* dst)
{
    __shared__ Box6 s_box[kBlock / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            box.lo[k] = min_nan(box.lo[k], __shfl_xor(box.lo[k], off, 64));
            box.hi[k] = max_nan(box.hi[k], __shfl_xor(box.hi[k], off, 64));
        }
    if ((threadIdx.x & 63) == 0) s_box[threadIdx.x >> 6] = box;
    __syncthreads();
    if (threadIdx.x < 3)
    {
        const int k = threadIdx.x;
        float lo = s_box[0].lo[k], hi = s_box[0].hi[k];
        for (int w = 1; w < kBlock / 64; ++w)
        {
            lo = min_nan(lo, s_box[w].lo[k]);
            hi = max_nan(hi, s_box[w].hi[k]);
        }
        dst[k]     = lo;
        dst[3 + k] = hi;
    }
}

__global__ __launch_bounds__(kBlock) void box_partial_kernel(const float4* __restrict__ position, int n,
                                                             float* __restrict__ partial)
{
    Box6 box = empty_box();
    const size_t step = (size_t)gridDim.x * kBlock;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < (size_t)n; i += step)
    {
        const float4 p = nt_load4(position + i);
        const float v[3] = {p.x, p.y, p.z};
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            box.lo[k] = min_nan(box.lo[k], v[k]);
            box.hi[k] = max_nan(box.hi[k], v[k]);
        }
    }
    box_of_block(box, partial + 6 * (size_t)blockIdx.x);
}

// out[0..5]: the box; out[6..11]: the mean of the partial boxes.  A far outlier stretches the box but only one of the
// partial ones: the two together say whether the box stands for the cloud.
__global__ __launch_bounds__(kBlock) void box_final_kernel(const float* __restrict__ partial, int blocks,
                                                           float* __restrict__ out)
{
    __shared__ float s_sum[kBlock / 64][6];
    Box6 box     = empty_box();
    float sum[6] = {0, 0, 0, 0, 0, 0};
    for (int i = threadIdx.x; i < blocks; i += kBlock)
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            const float lo = partial[6 * i + k], hi = partial[6 * i + 3 + k];
            box.lo[k] = min_nan(box.lo[k], lo);
            box.hi[k] = max_nan(box.hi[k], hi);
            sum[k] += lo;
            sum[3 + k] += hi;
        }
#pragma unroll
    for (int k = 0; k < 6; ++k)
    {
        sum[k] = wave_sum(sum[k]);
        if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6][k] = sum[k];
    }
    box_of_block(box, out);  // (its barrier is behind s_sum too)
    if (threadIdx.x < 6)
    {
        float all = 0.f;
        for (int w = 0; w < kBlock / 64; ++w) all += s_sum[w][threadIdx.x];
        out[6 + threadIdx.x] = all / (float)blocks;
    }
}

// ---- permutations -----------------------------------------------------------------------------------------------
// One row of 16 bytes per lane, four rows per thread: all index loads, then all gathers are in flight before anything
// waits.  What bounds it is the number of 64-byte lines the random rows touch: 10 M random rows take 0.3 ms, where
// torch's gather of the same rows, one row per wavefront's share of 16 bytes, takes 2.1 ms.  An index that names no
// row gives zeros.
constexpr int kGatherPer = 4;

__global__ __launch_bounds__(kBlock) void gather_rows_kernel(const float4* __restrict__ src, int rows,
                                                             const long long* __restrict__ index, int n,
                                                             float4* __restrict__ dst)
{
    const size_t base = (size_t)blockIdx.x * (kBlock * kGatherPer) + threadIdx.x;
    long long o[kGatherPer];
#pragma unroll
    for (int k = 0; k < kGatherPer; ++k)
    {
        const size_t i = base + k * kBlock;
        o[k]           = i < (size_t)n ? __builtin_nontemporal_load(index + i) : 0;
    }
    float4 v[kGatherPer];
#pragma unroll
    for (int k = 0; k < kGatherPer; ++k)
    {
        v[k] = make_float4(0, 0, 0, 0);
        if (base + k * kBlock < (size_t)n && (unsigned long long)o[k] < (unsigned long long)rows) v[k] = src[o[k]];
    }
#pragma unroll
    for (int k = 0; k < kGatherPer; ++k)
        if (base + k * kBlock < (size_t)n) nt_store4(dst + base + k * kBlock, v[k]);
}

// The cloud along `order` (a permutation), its blocks of `block` points shuffled: point i of the result is point
// order[perm[i / block] * block + i % block], the points behind the last whole block stay where `order` puts them.
// One pass in place of composing the two permutations and gathering by the result; the ids of the points and their
// normals come along.  10 M points in random order: 414 us, 20 M random lines (positions and normals).
__global__ __launch_bounds__(kBlock) void shuffle_gather_kernel(const float4* __restrict__ position,
                                                                const int32_t* __restrict__ normal,
                                                                const long long* __restrict__ order,
                                                                const long long* __restrict__ perm, int n, int block,
                                                                float4* __restrict__ out_position,
                                                                int32_t* __restrict__ out_normal,
                                                                int32_t* __restrict__ out_id)
{
    const size_t base = (size_t)blockIdx.x * (kBlock * kGatherPer) + threadIdx.x;
    const uint32_t whole = (uint32_t)(n / block) * (uint32_t)block;
    long long o[kGatherPer];
#pragma unroll
    for (int k = 0; k < kGatherPer; ++k)
    {
        const size_t i = base + k * kBlock;
        o[k]           = 0;
        if (i < (size_t)n)
        {
            size_t slot = i;
            if ((uint32_t)i < whole)
            {
                const uint32_t b = (uint32_t)i / (uint32_t)block;
                slot             = (size_t)perm[b] * (size_t)block + ((uint32_t)i - b * (uint32_t)block);
                if (slot >= (size_t)n) slot = i;  // (not a permutation)
            }
            o[k] = __builtin_nontemporal_load(order + slot);
        }
    }
    float4 v[kGatherPer];
    int32_t m[kGatherPer];
#pragma unroll
    for (int k = 0; k < kGatherPer; ++k)
    {
        v[k] = make_float4(0, 0, 0, 0);
        m[k] = 0;
        if (base + k * kBlock < (size_t)n && (unsigned long long)o[k] < (unsigned long long)n)
        {
            v[k] = position[o[k]];
            if (normal) m[k] = normal[o[k]];
        }
    }
#pragma unroll
    for (int k = 0; k < kGatherPer; ++k)
    {
        const size_t i = base + k * kBlock;
        if (i < (size_t)n)
        {
            nt_store4(out_position + i, v[k]);
            if (normal) __builtin_nontemporal_store(m[k], out_normal + i);
            __builtin_nontemporal_store((int32_t)o[k], out_id + i);
        }
    }
}

// ---- radii and the order inside the blocks ----------------------------------------------------------------------
// ComputeRadius (SceneData.cpp:462-483) from the neighbour distance and the uniform number of every point, then
// SortBlocksByRadius (:671-684) for blocks of kBlock points, one workgroup each: the (radius, slot) keys of a block
// are sorted in registers, 33 of the 36 steps of the bitonic network between lanes of a wavefront, 3 through LDS, and
// the rows of the block are written in that order.  10 M points: 146 us for 840 MB, 5.8 TB/s, in place of a segmented
// sort (464 us), two gathers and eight elementwise passes.  The slot in the low word makes the sort stable; a radius
// that is not a number comes last.  The points behind the last whole block keep their order.
__global__ __launch_bounds__(kBlock) void radius_blocks_kernel(const float4* __restrict__ position,
                                                               const int32_t* __restrict__ normal,
                                                               const int32_t* __restrict__ id,
                                                               const float* __restrict__ distance,
                                                               const double* __restrict__ uniform, int n,
                                                               float4* __restrict__ out_position,
                                                               int32_t* __restrict__ out_normal,
                                                               float4* __restrict__ out_data,
                                                               long long* __restrict__ out_order)
{
    __shared__ unsigned long long s_key[kBlock];
    __shared__ float s_d[kBlock], s_s[kBlock];
    const int t       = threadIdx.x;
    const size_t row0 = (size_t)blockIdx.x * kBlock;
    const size_t i    = row0 + t;
    float r           = 0.f;
    if (i < (size_t)n)
    {
        const float d  = __builtin_nontemporal_load(distance + i);
        const double u = __builtin_nontemporal_load(uniform + i);
        const float s  = (float)sqrt(1.0 / (u < 1e-300 ? 1e-300 : u));
        s_d[t]         = d;
        s_s[t]         = s;
        r              = d * s;
    }
    // ascending keys: sign-magnitude floats as ordered words
    const uint32_t bits = __float_as_uint(r);
    uint32_t ordered    = (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
    if (r != r) ordered = 0xFFFFFFFFu;
    unsigned long long key = (unsigned long long)ordered << 32 | (uint32_t)t;
    const bool sorted = row0 + kBlock <= (size_t)n;  // (workgroup-uniform)
    if (sorted)
    {
#pragma unroll
        for (int k = 2; k <= kBlock; k <<= 1)
#pragma unroll
            for (int j = k >> 1; j > 0; j >>= 1)
            {
                unsigned long long other;
                if (j >= 64)
                {
                    __syncthreads();
                    s_key[t] = key;
                    __syncthreads();
                    other = s_key[t ^ j];
                }
                else
                    other = __shfl_xor(key, j, 64);
                const bool keep_small = ((t & k) == 0) == ((t & j) == 0);
                key                   = (other < key) == keep_small ? other : key;
            }
    }
    __syncthreads();  // s_d and s_s are complete
    if (i >= (size_t)n) return;
    const int q     = (int)(uint32_t)key;
    const size_t at = row0 + q;
    const float d = s_d[q], s = s_s[q];
    const float rad = d * s;
    float4 p        = position[at];
    p.w             = rad;
    nt_store4(out_position + i, p);
    nt_store4(out_data + i, make_float4(d, 0.f, s, rad));
    if (normal) __builtin_nontemporal_store(normal[at], out_normal + i);
    __builtin_nontemporal_store((long long)id[at], out_order + i);
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
size_t bounding_box_floats() { return 6 * (size_t)(kBoxBlocks + 2); }

void launch_bounding_box(const float4* position, int n, float* box, hipStream_t st)
{
    const int want   = (n + kBlock * 4 - 1) / (kBlock * 4);
    const int blocks = want < 1 ? 1 : (want < kBoxBlocks ? want : kBoxBlocks);
    hipLaunchKernelGGL(box_partial_kernel, dim3(blocks), dim3(kBlock), 0, st, position, n, box + 12);
    hipLaunchKernelGGL(box_final_kernel, dim3(1), dim3(kBlock), 0, st, box + 12, blocks, box);
}

static int gather_blocks(int n) { return (int)(((size_t)n + kBlock * kGatherPer - 1) / (kBlock * kGatherPer)); }

void launch_gather_rows(const float4* src, int rows, const long long* index, int n, float4* dst, hipStream_t st)
{
    hipLaunchKernelGGL(gather_rows_kernel, dim3(gather_blocks(n)), dim3(kBlock), 0, st, src, rows, index, n, dst);
}

void launch_shuffle_gather(const float4* position, const int32_t* normal, const long long* order, const long long* perm,
                           int n, int block, float4* out_position, int32_t* out_normal, int32_t* out_id, hipStream_t st)
{
    hipLaunchKernelGGL(shuffle_gather_kernel, dim3(gather_blocks(n)), dim3(kBlock), 0, st, position, normal, order, perm, n,
                       block, out_position, out_normal, out_id);
}

void launch_radius_blocks(const float4* position, const int32_t* normal, const int32_t* id, const float* distance,
                          const double* uniform, int n, float4* out_position, int32_t* out_normal, float4* out_data,
                          long long* out_order, hipStream_t st)
{
    hipLaunchKernelGGL(radius_blocks_kernel, dim3((int)(((size_t)n + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, position,
                       normal, id, distance, uniform, n, out_position, out_normal, out_data, out_order);
}

}  // namespace adop
