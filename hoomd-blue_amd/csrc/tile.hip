// tile.hip -- neighbour-list build over columns of cells (tile.h).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kernel_util.h"
#include "tile.h"

namespace hm
{

constexpr unsigned int COL_BLOCK = 256;
constexpr unsigned int COL_PAD = 32;         // readable entries after the staged particles

bool choose_columns(unsigned int N, const unsigned int dim[3], ColGeom& g)
{
    if (N == 0 || dim[0] < 4 || dim[1] < 4 || dim[2] < 4)
        return false;
    const double ncol = (double)dim[0] * dim[1], mean = N / (ncol * dim[2]);
    // Taller columns stage fewer shell layers per home layer; short ones keep enough workgroups in
    // flight (about 2 000) and their LDS small (a column of about 1 200 staged particles).
    unsigned int h = (unsigned int)std::max(1.0, std::floor(ncol * dim[2] / 2048.0));
    h = std::min(h, (unsigned int)std::max(1.0, std::floor(1200.0 / (9.0 * mean) - 2.0)));
    h = std::min(std::min(h, COL_Z), dim[2] - 3);  // the staged span stays below half the box
    g.nz = (dim[2] + h - 1) / h;
    const unsigned int tallest = (dim[2] + g.nz - 1) / g.nz;
    g.ntile = dim[0] * dim[1] * g.nz;
    const double st = mean * 9.0 * (tallest + 2.0);
    const double cap = st * 1.25 + 4.0 * std::sqrt(st) + 64.0;
    g.cap = (unsigned int)(std::ceil(cap / 64.0) * 64.0);  // at most 1 728 at 8 a cell: 28 KB
    g.hcap = g.cap / 4;
    g.lpc = 4;
    while (g.lpc < 32 && g.lpc < mean * 1.2)
        g.lpc *= 2;
    g.group = 27.0 * mean <= 112.0 ? 4 : 8;
    g.dmax = 0.5f * tallest + 1.0f;
    return true;
}

struct ColIndex
{
    unsigned int cid[COL_CELLS];      // cell of each staged cell
    unsigned int off[COL_CELLS + 1];  // first staged particle of each staged cell
    float4 shift[COL_CELLS];          // offset of each staged cell's origin from the column centre; code in w
    unsigned int hoff[COL_Z + 1];     // first home ordinal of each home cell
};

__device__ __forceinline__ unsigned int wave_prefix(unsigned int v, unsigned int lane)
{
#pragma unroll
    for (unsigned int o = 1; o < 64; o <<= 1)
    {
        const unsigned int u = __shfl_up(v, o, 64);
        if (lane >= o)
            v += u;
    }
    return v;
}

// One neighbour test shifted into the low end of mask m: the sign of t. A t of zero, whose sign says
// nothing, lies in every guard band. One v_alignbit; a compare into VCC and an add with carry would need
// two wait states between them on gfx950.
__device__ __forceinline__ void push_hit(unsigned int& m, float t)
{
    m = __builtin_amdgcn_alignbit(m, __float_as_uint(t), 31);
}

// place (0, 1, 2) of offset o among the neighbours h - 1, h, h + 1 sorted by wrapped coordinate; rank is
// the place of offset 0 (sorted_neighbour's order)
__device__ __forceinline__ unsigned int sorted_place(int o, unsigned int rank)
{
    return (unsigned int)(o + (int)rank + 3) % 3u;
}

// One home particle's row when the column's particles do not fit the stage: its 27 cells from memory,
// the FP64 test of every candidate. Called by the G lanes of a group together; the other groups of
// the wavefront may take other trip counts, so the lanes exchange hits by shuffles within the group.
template<int G, bool MT, bool EXCL, bool SLOT>
__device__ __forceinline__ void unstaged_row(const NlistKernelArgs& a, const ColIndex& S, int hx, int hy,
                                          int z0, unsigned int nh, unsigned int mid, unsigned int h,
                                          unsigned int sub)
{
#pragma clang fp contract(off)
    unsigned int hz = 0;
    while (hz + 1 < nh && S.hoff[hz + 1] <= h)
        hz++;
    const size_t hs = (size_t)S.cid[9 * (hz + 1) + mid] * a.cmax + (h - S.hoff[hz]);
    const unsigned int i = a.srel ? a.sidx[hs] : a.entries[hs].idx;
    const double4 pi = a.pos[i];
    const unsigned int ti = MT ? (unsigned int)pi.w : 0u;
    unsigned int ex[4] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0xffffffffu};
    if (EXCL)
        load_exclusions(a, i, ex[0], ex[1], ex[2], ex[3]);
    unsigned int cnt = 0;
    for (int q = 0; q < 27; q++)
    {
        int x, y, z;
        const int ox = sorted_neighbour(hx, (int)a.dim[0], q % 3, x);
        const int oy = sorted_neighbour(hy, (int)a.dim[1], (q / 3) % 3, y);
        const int oz = sorted_neighbour(z0 + (int)hz, (int)a.dim[2], q / 9, z);
        const unsigned int id = (unsigned int)(x + (int)a.dim[0] * (y + (int)a.dim[1] * z));
        const unsigned int n = min(a.cell_size[id], a.cmax);
        for (unsigned int b = 0; b < n; b += G)
        {
            bool hit = false;
            unsigned int e = 0;
            if (b + sub < n)
            {
                const size_t sl = (size_t)id * a.cmax + b + sub;
                const unsigned int j = a.srel ? a.sidx[sl] : a.entries[sl].idx;
                const double4 pj = a.pos[j];
                double qx = pi.x - pj.x, qy = pi.y - pj.y, qz = pi.z - pj.z;
                min_image(a.box, qx, qy, qz);
                const unsigned int tp = MT ? ti * a.ntypes + (unsigned int)pj.w : 0u;
                hit = j != i && a.enabled[tp] && qx * qx + qy * qy + qz * qz <= a.rlistsq[tp];
                if (EXCL)
                    hit = hit && j != ex[0] && j != ex[1] && j != ex[2] && j != ex[3];
                e = SLOT ? (unsigned int)sl | offset_code(-ox, -oy, -oz) : j;
            }
            unsigned int before = hit ? 1u : 0u;
#pragma unroll
            for (unsigned int o = 1; o < G; o <<= 1)
            {
                const unsigned int v = __shfl_up(before, o, G);
                if (sub >= o)
                    before += v;
            }
            const unsigned int at = cnt + before - 1u;
            if (hit && at < a.nmax)
                a.nlist[(size_t)i * a.nmax + (SLOT ? row_store_pos(at) : at)] = e;
            cnt += __shfl(before, G - 1, G);
        }
    }
    if (sub == 0)
    {
        a.n_neigh[i] = cnt;
        if (cnt > a.nmax)
            atomicMax(a.cond, cnt);
    }
}

// Home particle of a column: particle index; staged position | home layer << 16 | type << 24
struct ColHome
{
    unsigned int i, at;
};

// Neighbour rows of a column where cells hold a few particles, G lanes per home particle. The
// candidates are one run of LDS; each lane tests its own contiguous part of it, 32 candidates at a
// time: three differences, three multiply-adds that end at r^2 - r_list^2, a running minimum of its
// magnitude for the guard band, and the hit bit (about ten vector instructions and one LDS read per
// 64 tests, no ballot). A prefix sum of the lanes' hit counts places each lane's hits in the row, so
// rows stay in candidate order. Candidates in the guard band take the CPU's FP64 decision. SLOT: row
// entries are cell slots with offset codes in transposed blocks (pair_rel_kernel's rows), else
// particle indices.
//
// The one-wavefront-per-cell form stages 27 cells for every home cell of about three particles and compacts
// every 64 tests by ballot (about 765 vector instructions per cell). 10^6 beads of a melt, 3.0 a cell, 12.5
// neighbours, exclusions: 370 us a build, that form 553. Waves wait 70 % of their cycles (SQ_WAIT_ANY 619 M
// of 882 M); the 200 MB it reads and 135 MB it writes would take 70 us, its 114 M vector instructions 190
// (four cycles each on 1 024 SIMDs): what bounds it is the chain of each column (cell sizes, staging, rows)
// with five to seven workgroups per CU in flight.
template<int G, bool MT, bool EXCL, bool SLOT>
__global__ __launch_bounds__(COL_BLOCK) void nlist_col_kernel(NlistKernelArgs a, ColGeom g)
{
#pragma clang fp contract(off)
    extern __shared__ float4 sc[];  // offset from the column centre, row entry in w
    __shared__ ColIndex S;
    ColHome* const home = (ColHome*)(sc + g.cap + COL_PAD);
    ushort4* const hex = (ushort4*)(home + g.hcap);  // staged positions of each home's exclusions
    unsigned char* const stype = (unsigned char*)(hex + (EXCL ? g.hcap : 0));
    if (gate_closed(a.gate))
        return;
    count_build(a);
    const unsigned int tid = threadIdx.x, lane = tid & 63u;
    const unsigned int sgrp = tid / g.lpc, ssub = tid % g.lpc, nsgrp = COL_BLOCK / g.lpc;
    const unsigned int sub = tid % G;
    const int dx = (int)a.dim[0], dy = (int)a.dim[1], dz = (int)a.dim[2];
    const XcdRange r = xcd_range(g.ntile);
    for (unsigned int tile = r.begin; tile < r.end; tile += r.stride)
    {
        const int hx = (int)(tile % a.dim[0]), hy = (int)((tile / a.dim[0]) % a.dim[1]);
        const unsigned int zt = tile / (a.dim[0] * a.dim[1]);
        const int z0 = (int)(zt * a.dim[2] / g.nz), z1 = (int)((zt + 1) * a.dim[2] / g.nz);
        const unsigned int nh = (unsigned int)(z1 - z0), nsc = 9 * (nh + 2);
        // place of the home column among the nine of a layer
        const unsigned int rx = hx == 0 ? 0u : (hx == dx - 1 ? 2u : 1u),
                           ry = hy == 0 ? 0u : (hy == dy - 1 ? 2u : 1u), mid = rx + 3u * ry;
        if (tid < 64)
        {
            unsigned int carry = 0;
            for (unsigned int q0 = 0; q0 < nsc; q0 += 64)
            {
                const unsigned int q = q0 + lane;
                unsigned int sz = 0;
                if (q < nsc)
                {
                    const unsigned int c9 = q % 9u;
                    const int layer = (int)(q / 9u);
                    int x, y, z = z0 - 1 + layer;
                    const int ox = sorted_neighbour(hx, dx, (int)(c9 % 3u), x);
                    const int oy = sorted_neighbour(hy, dy, (int)(c9 / 3u), y);
                    z += z < 0 ? dz : (z >= dz ? -dz : 0);
                    const unsigned int id = (unsigned int)(x + dx * (y + dy * z));
                    S.cid[q] = id;
                    S.shift[q] = make_float4(((float)ox - 0.5f) * a.cwf[0], ((float)oy - 0.5f) * a.cwf[1],
                                             ((float)layer - 1.f - 0.5f * nh) * a.cwf[2],
                                             // x and y offsets; minus the layer in the two z bits,
                                             // so that adding the home layer completes the code
                                             __uint_as_float(offset_code(-ox, -oy, -layer)));
                    sz = min(a.cell_size[id], a.cmax);
                }
                const unsigned int incl = wave_prefix(sz, lane);
                if (q < nsc)
                    S.off[q] = carry + incl - sz;
                carry += __shfl(incl, 63, 64);
            }
            if (lane == 0)
                S.off[nsc] = carry;
        }
        __syncthreads();
        if (tid < 64)
        {
            const unsigned int q = 9 * (lane + 1) + mid;
            const unsigned int n = lane < nh ? S.off[q + 1] - S.off[q] : 0u;
            const unsigned int incl = wave_prefix(n, lane);
            if (lane < nh)
                S.hoff[lane] = incl - n;
            if (lane == nh - 1)
                S.hoff[nh] = incl;
        }
        const double wz = a.box.L[2] / (double)a.dim[2];
        const double cx = a.box.lo[0] + (hx + 0.5) * (a.box.L[0] / (double)a.dim[0]);
        const double cy = a.box.lo[1] + (hy + 0.5) * (a.box.L[1] / (double)a.dim[1]);
        const double cz = a.box.lo[2] + (z0 + 0.5 * nh) * wz;
        __syncthreads();
        const unsigned int total = S.off[nsc], nhome = S.hoff[nh];
        const bool fits = total <= g.cap && nhome <= g.hcap;
        if (!fits && a.crowded && tid == 0)
            atomicAdd(a.crowded, nhome);
        if (fits)
            for (unsigned int q = sgrp; q < nsc; q += nsgrp)
            {
                const unsigned int o = S.off[q], n = S.off[q + 1] - o;
                const size_t base = (size_t)S.cid[q] * a.cmax;
                const float4 sh = S.shift[q];
                const unsigned int layer = q / 9u;
                const bool own = q % 9u == mid && layer > 0 && layer <= nh;
                for (unsigned int k = ssub; k < n; k += g.lpc)
                {
                    float3 p;
                    unsigned int j, type = 0;
                    if (a.srel)
                    {
                        const float3 rr = a.srel[base + k];
                        p = make_float3(rr.x + sh.x, rr.y + sh.y, rr.z + sh.z);
                        j = (!SLOT || own) ? a.sidx[base + k] : 0u;
                        if (MT)
                            type = a.swrd[base + k] >> 24;
                    }
                    else
                    {
                        const hm_cell_entry ce = a.entries[base + k];
                        p = rel_to_centre(a.box, ce.x, ce.y, ce.z, cx, cy, cz);
                        j = ce.idx;
                        type = ce.type;
                    }
                    sc[o + k] = make_float4(p.x, p.y, p.z,
                                            SLOT ? __uint_as_float((unsigned int)(base + k) | __float_as_uint(sh.w))
                                                 : __uint_as_float(j));
                    if (MT)
                        stype[o + k] = (unsigned char)type;
                    if (own)
                    {
                        const unsigned int h = S.hoff[layer - 1] + k;
                        home[h] = ColHome{j, (o + k) | ((layer - 1) << 16) | (type << 24)};
                        if (EXCL)
                        {
                            unsigned int x[4] = {NO_SLOT, NO_SLOT, NO_SLOT, NO_SLOT};
                            load_exclusions(a, j, x[0], x[1], x[2], x[3]);
                            unsigned short at[4];
#pragma unroll
                            for (int e = 0; e < 4; e++)
                            {
                                at[e] = 0xffffu;
                                if (x[e] == NO_SLOT)
                                    continue;
                                // the excluded particle's cell, if it is one of the 27, and its place
                                const unsigned int sl = a.slot_of[x[e]], c = sl / a.cmax;
                                const int ex = wrap_offset((int)(c % a.dim[0]) - hx, dx);
                                const int ey = wrap_offset((int)((c / a.dim[0]) % a.dim[1]) - hy, dy);
                                const int ez = wrap_offset((int)(c / (a.dim[0] * a.dim[1])) - (z0 + (int)layer - 1), dz);
                                if (ex < -1 || ex > 1 || ey < -1 || ey > 1 || ez < -1 || ez > 1)
                                    continue;
                                const unsigned int px = sorted_place(ex, rx), py = sorted_place(ey, ry);
                                const unsigned int eq = 9u * (unsigned int)((int)layer + ez) + 3u * py + px;
                                at[e] = (unsigned short)(S.off[eq] + (sl - c * a.cmax));
                            }
                            hex[h] = make_ushort4(at[0], at[1], at[2], at[3]);
                        }
                    }
                }
            }
        __syncthreads();
        for (unsigned int h0 = 0; h0 < nhome; h0 += COL_BLOCK / G)
        {
            const unsigned int h = h0 + tid / G;
            const bool active = h < nhome;
            if (!fits)
            {
                if (active)
                    unstaged_row<G, MT, EXCL, SLOT>(a, S, hx, hy, z0, nh, mid, h, sub);
                continue;
            }
            const ColHome hm = home[active ? h : 0u];
            const unsigned int i = hm.i, self = hm.at & 0xffffu, hz = (hm.at >> 16) & 0xffu,
                               ti = MT ? hm.at >> 24 : 0u;
            ushort4 ex = make_ushort4(0xffffu, 0xffffu, 0xffffu, 0xffffu);
            if (EXCL)
                ex = hex[active ? h : 0u];
            const float4 me = sc[self];
            // r_list^2 of each candidate type (negative for a disabled pair: never a hit)
            float rl[MT ? HM_MAX_TYPES : 1];
            float guard = 0.f;
#pragma unroll
            for (unsigned int t = 0; t < (MT ? HM_MAX_TYPES : 1); t++)
            {
                const unsigned int tp = MT ? ti * a.ntypes + (t < a.ntypes ? t : 0u) : 0u;
                rl[t] = a.enabled[tp] ? a.rlistsq_f[tp] : -1.f;
                guard = fmaxf(guard, a.guard[tp]);
            }
            auto test = [&](unsigned int k) {
                const float4 p = sc[k];
                float l = rl[0];
                if (MT)
                {
                    const unsigned int tj = stype[k];
                    l = tj == 1u ? rl[MT ? 1 : 0] : (tj == 2u ? rl[MT ? 2 : 0] : (tj == 3u ? rl[MT ? 3 : 0] : l));
                }
                const float qx = me.x - p.x, qy = me.y - p.y, qz = me.z - p.z;
                return fmaf(qx, qx, fmaf(qy, qy, fmaf(qz, qz, -l)));
            };
            unsigned int* const row = a.nlist + (size_t)i * a.nmax;
            const unsigned int zadd = SLOT ? (hz + 1) << 30 : 0u;
            unsigned int cnt = 0;
            // candidates [b, e) split over the group's lanes in order
            auto sweep = [&](unsigned int b, unsigned int e) {
                const unsigned int len = (e - b + G - 1) / G;
                const unsigned int k = min(b + sub * len, e);
                const unsigned int end = min(k + len, e);
                unsigned int m = 0;
                float mn = 3e38f;
#pragma unroll
                for (unsigned int t = 0; t < 32; t += 4)
                {
                    if (t != 0 && !wave_ballot(k + t < end))
                    {
                        m <<= 32 - t;
                        break;
                    }
                    float d[4];
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        d[u] = test(k + t + u);
#pragma unroll
                    for (int u = 0; u < 4; u++)
                    {
                        mn = fminf(mn, fabsf(d[u]));
                        push_hit(m, d[u]);
                    }
                }
                const unsigned int left = end - k;
                if (mn <= guard)
                    // a candidate inside the guard band: the FP64 decision as
                    // NeighborListBinned.cc:151-157 computes it
                    for (unsigned int t = 0; t < min(left, 32u); t++)
                        if (fabsf(test(k + t)) <= guard)
                        {
                            const unsigned int w = __float_as_uint(sc[k + t].w), bit = 0x80000000u >> t;
                            const unsigned int tp = MT ? ti * a.ntypes + stype[k + t] : 0u;
                            const double4 pi = a.pos[i], pj = a.pos[SLOT ? a.sidx[w & OFFSET_CODE_MASK] : w];
                            double qx = pi.x - pj.x, qy = pi.y - pj.y, qz = pi.z - pj.z;
                            min_image(a.box, qx, qy, qz);
                            m = qx * qx + qy * qy + qz * qz <= a.rlistsq[tp] && a.enabled[tp] ? m | bit : m & ~bit;
                        }
                if (left < 32)
                    m &= ~(0xffffffffu >> left);
                auto drop = [&](unsigned int at) {
                    if (at - k < 32)
                        m &= ~(0x80000000u >> (at - k));
                };
                drop(self);
                if (EXCL)
                {
                    drop(ex.x);
                    drop(ex.y);
                    if (a.max_excl > 2)
                    {
                        drop(ex.z);
                        drop(ex.w);
                    }
                }
                unsigned int incl = (unsigned int)__popc(m);
                const unsigned int mine = incl;
#pragma unroll
                for (unsigned int o = 1; o < G; o <<= 1)
                {
                    const unsigned int v = __shfl_up(incl, o, G);
                    if (sub >= o)
                        incl += v;
                }
                unsigned int p = cnt + incl - mine;
                cnt += __shfl(incl, G - 1, G);
                while (wave_ballot(m != 0))
                    if (m)
                    {
                        const unsigned int t = (unsigned int)__clz((int)m);
                        m &= ~(0x80000000u >> t);
                        if (p < a.nmax)
                            row[SLOT ? row_store_pos(p) : p] = __float_as_uint(sc[k + t].w) + zadd;
                        p++;
                    }
            };
            const int gz = z0 + (int)hz;
            unsigned int l0 = S.off[9 * hz], l3 = S.off[9 * hz + 27], c = l0;
            if (gz == 0)  // the run is cut by the wrap of z
                c = S.off[9 * hz + 9];
            else if (gz == dz - 1)
                c = S.off[9 * hz + 18];
            if (!active)
                l0 = l3 = c = 0;
            // at most 32 G candidates a sweep, so that a lane's part is one word
            auto run = [&](unsigned int b, unsigned int e) {
                for (; wave_ballot(b < e); b = min(b + 32 * G, e))
                    sweep(b, min(b + 32 * G, e));
            };
            run(c, l3);
            if (wave_ballot(c != l0))
                run(l0, c);
            if (active && sub == 0)
            {
                a.n_neigh[i] = cnt;
                if (cnt > a.nmax)
                    atomicMax(a.cond, cnt);
            }
        }
        __syncthreads();
    }
}

template<int G, bool MT, bool EXCL>
static void col_dispatch(const NlistKernelArgs& a, const ColGeom& g, unsigned int grid,
                         unsigned int lds, hipStream_t s)
{
    if (a.offset_codes)
        hipLaunchKernelGGL((nlist_col_kernel<G, MT, EXCL, true>), dim3(grid), dim3(COL_BLOCK), lds,
                           s, a, g);
    else
        hipLaunchKernelGGL((nlist_col_kernel<G, MT, EXCL, false>), dim3(grid), dim3(COL_BLOCK),
                           lds, s, a, g);
}

template<int G>
static void col_dispatch_types(const NlistKernelArgs& a, const ColGeom& g, unsigned int grid,
                               unsigned int lds, hipStream_t s)
{
    const bool mt = a.ntypes > 1, ex = a.n_excl != nullptr && a.max_excl > 0;
    if (mt)
        ex ? col_dispatch<G, true, true>(a, g, grid, lds, s)
           : col_dispatch<G, true, false>(a, g, grid, lds, s);
    else
        ex ? col_dispatch<G, false, true>(a, g, grid, lds, s)
           : col_dispatch<G, false, false>(a, g, grid, lds, s);
}

hipError_t launch_nlist_columns(const NlistKernelArgs& a_in, const ColGeom& g, hipStream_t s)
{
    NlistKernelArgs a = a_in;
    const double u = 1.0 / 16777216.0;
    double wmax = 0.0;
    for (int d = 0; d < 3; d++)
        wmax = fmax(wmax, a.box.L[d] / (double)a.dim[d]);
    // FP32 error of a coordinate difference, in units of u w, for coordinates within D = dmax cells
    // of the column centre. From entries: each coordinate rounded once (D, twice) and the
    // difference, about one cell near the threshold, once (2). From the relative positions: the
    // position (1), the FP32 width times the offset (2 D) and the sum (D), twice, and the difference.
    const double D = g.dmax;
    const double e_dx = u * wmax * (a.srel ? 2.0 * (1.0 + 3.0 * D) + 2.0 : 2.0 * D + 2.0);
    const unsigned int nt = a.ntypes ? a.ntypes : 1;
    for (unsigned int q = 0; q < nt * nt; q++)
    {
        const double rl2 = a.rlistsq[q];
        a.rlistsq_f[q] = (float)rl2;
        a.guard[q] = (float)(4.0 * (2.0 * sqrt(3.0) * sqrt(rl2) * e_dx + 6.0 * u * rl2) + 1e-12);
    }
    const unsigned int grid = round_up(min(g.ntile, GATED_BLOCKS), 8);
    const bool ex = a.n_excl != nullptr && a.max_excl > 0;
    const unsigned int lds = (g.cap + COL_PAD) * (unsigned int)sizeof(float4)
                             + g.hcap * (unsigned int)(sizeof(ColHome) + (ex ? sizeof(ushort4) : 0))
                             + (a.ntypes > 1 ? g.cap + COL_PAD : 0);
    if (g.group == 4)
        col_dispatch_types<4>(a, g, grid, lds, s);
    else
        col_dispatch_types<8>(a, g, grid, lds, s);
    return hipGetLastError();
}

} // namespace hm
