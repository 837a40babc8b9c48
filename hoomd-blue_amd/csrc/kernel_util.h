// kernel_util.h -- device helpers shared by the kernel sources: gated persistent grids, sorted cell
// neighbours, list-build building blocks.
#pragma once

#include "kernels.h"

namespace hm
{

// ======================================================================== persistent grids
// Kernels that only run on a neighbour-list rebuild are launched every step and exit at once
// when the device-side rebuild flag is not set. They walk their work in grid-stride loops over a
// bounded grid, so an idle step costs a few hundred empty workgroups instead of one per cell.
constexpr unsigned int GATED_BLOCKS = 2048;

__device__ __forceinline__ bool gate_closed(const StepState* gate)
{
    return gate && gate->rebuild_at != gate->timestep + 1;
}

// XCD-aware persistent loop: workgroup b runs on XCD (b % 8); it visits the items of that XCD's
// contiguous eighth of [0, n) with stride gridDim.x / 8.
struct XcdRange
{
    unsigned int begin, end, stride;
};

__device__ __forceinline__ XcdRange xcd_range(unsigned int n)
{
    const unsigned int xcd = blockIdx.x & 7u, r = blockIdx.x >> 3, per = gridDim.x >> 3;
    const unsigned int chunk = (n + 7) / 8;
    XcdRange x;
    x.begin = xcd * chunk + r;
    x.end = min(n, (xcd + 1) * chunk);
    x.stride = per;
    return x;
}

// The k-th smallest (k = 0, 1, 2) of the wrapped coordinates h - 1, h, h + 1 on an axis of
// d >= 3 cells; returns its offset from h and sets n to the coordinate.
__device__ __forceinline__ int sorted_neighbour(int h, int d, int k, int& n)
{
    int off;
    if (h == 0)  // h - 1 wraps to d - 1, the largest
        off = k == 0 ? 0 : (k == 1 ? 1 : -1);
    else if (h == d - 1)  // h + 1 wraps to 0, the smallest
        off = k == 0 ? 1 : (k == 1 ? -1 : 0);
    else
        off = k - 1;
    n = h + off;
    if (n < 0)
        n += d;
    else if (n >= d)
        n -= d;
    return off;
}

// Minimum-image offset of a position from a centre, rounded to FP32. The caller keeps every staged particle
// inside half a box of it: within 1.5 cell widths of a cell's centre on grids of 4 cells or more, within
// half a column and one layer of a column's (up to 9 cell widths; choose_columns).
__device__ __forceinline__ float3 rel_to_centre(const DevBox& b, double x, double y, double z,
                                                double cx, double cy, double cz)
{
#pragma clang fp contract(off)
    double dx = x - cx, dy = y - cy, dz = z - cz;
    min_image(b, dx, dy, dz);
    return make_float3((float)dx, (float)dy, (float)dz);
}

__device__ __forceinline__ void load_exclusions(const NlistKernelArgs& a, unsigned int i,
                                                unsigned int& ex0, unsigned int& ex1,
                                                unsigned int& ex2, unsigned int& ex3)
{
    unsigned int ne = min(a.n_excl[i], a.max_excl);
    const unsigned int* er = a.excl + (size_t)i * a.max_excl;
    if (ne > 0)
        ex0 = er[0];
    if (ne > 1)
        ex1 = er[1];
    if (ne > 2)
        ex2 = er[2];
    if (ne > 3)
        ex3 = er[3];
}

// Build statistics of NeighborList::needsUpdating (NeighborList.cc:1349-1415), kept by one thread
// of an open build.
__device__ __forceinline__ void count_build(const NlistKernelArgs& a)
{
    if (a.counter && blockIdx.x == 0 && threadIdx.x == 0)
    {
        StepState* st = a.counter;
        const unsigned long long t1 = st->timestep + 1;
        if (st->forced_at != t1)
        {
            if (t1 > st->last_update && t1 - st->last_update < st->shortest)
                st->shortest = t1 - st->last_update;
            if (a.dist_check && a.check_delay > 1 && t1 == st->last_update + a.check_delay)
                st->n_dangerous++;
        }
        st->last_update = t1;
        st->n_builds++;
    }
}

// The next slot of cell bin for every lane with ok, called by every lane of a wavefront in step; the
// active lanes must be its low lanes.
__device__ __forceinline__ unsigned int claim_slot(unsigned int bin, bool ok, unsigned int* cell_size)
{
    // slot allocation aggregated over runs of consecutive lanes in one cell (particles in
    // Hilbert order fill a cell from neighbouring indices): the first lane of a run adds the
    // run's length, and every run's atomic is issued by the one instruction. Active lanes are
    // the low lanes of the wave, so a lane's predecessor is active.
    const unsigned int lane = lane_id();
    const unsigned int prev = __shfl_up(bin, 1, 64);
    const bool head = ok && (lane == 0 || prev != bin || !__shfl_up((int)ok, 1, 64));
    const uint64_t heads = wave_ballot(head);
    // lanes that do not continue a run: heads, lanes not binned, inactive lanes
    const uint64_t stop = ~wave_ballot(ok && !head);
    const uint64_t upto = lane == 63 ? ~0ull : ((1ull << (lane + 1)) - 1ull);
    const unsigned int first = 63u - (unsigned int)__clzll((long long)(heads & upto));
    unsigned int base = 0;
    if (head)
    {
        const uint64_t after = lane == 63 ? 0ull : (stop >> (lane + 1));
        const unsigned int len = after ? (unsigned int)__ffsll((long long)after) : 64u - lane;
        base = atomicAdd(&cell_size[bin], len);
    }
    base = __shfl(base, (int)(ok ? first : lane), 64);
    return ok ? base + (lane - first) : 0u;
}

} // namespace hm
