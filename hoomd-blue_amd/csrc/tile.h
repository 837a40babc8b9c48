// tile.h -- columns of cells whose particles one workgroup owns.
//
// A column tile is up to COL_Z cells stacked along z. The workgroup stages the particles of the
// column and of the eight columns around it in LDS, layer by layer, the nine cells of a layer in
// increasing cell index. The candidates of a home particle (its 27 adjacent cells) are then three
// adjacent layers: one contiguous run of LDS, in the order of the reference's rows (two runs in
// the first and last cell of the axis, where the wrapped layer's cell index sorts differently).
#pragma once

#include "kernels.h"

namespace hm
{

constexpr unsigned int COL_Z = 16;                     // cells of a column, at most
constexpr unsigned int COL_CELLS = 9 * (COL_Z + 2);    // staged cells, at most

struct ColGeom
{
    unsigned int nz;       // columns along z: column k covers cells [k dz / nz, (k + 1) dz / nz)
    unsigned int ntile;    // dx dy nz
    unsigned int lpc;      // lanes that stage one cell (power of two)
    unsigned int cap;      // staged particles that fit the workgroup's LDS
    unsigned int hcap;     // home particles that fit it
    unsigned int group;    // lanes that share a home particle
    float dmax;            // largest distance of a staged cell's far face from the column centre, cells
};

// Column shape for N particles in dim cells; false where columns do not apply (fewer than 4 cells
// along an axis).
bool choose_columns(unsigned int N, const unsigned int dim[3], ColGeom& g);

hipError_t launch_nlist_columns(const NlistKernelArgs& a, const ColGeom& g, hipStream_t s);

} // namespace hm
