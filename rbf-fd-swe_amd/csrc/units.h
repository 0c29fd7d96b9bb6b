// Units of the matrix-core resident kernels (k_units.hip, k_units32.hip): the
// tables they share and the copy of a tile's rows.
//
// A workgroup owns one compact tile of consecutive nodes in a kernel order
// of its own, cut into units of 16 nodes; a wave takes whole units.  Lane
// 4 b + j of a unit ends up with node b, variable j.
#pragma once

#include "res_sync.h"

namespace swe {

// Where a launch keeps a unit's data between stages.
enum UnitMode {
    UM_RESIDENT,   // every unit's weights stay in registers
    UM_STREAM,     // R units per wave do, the others read theirs each stage;
                   // positions and the streamed units' H and D in LDS
    UM_GLOBAL      // the same with those units' positions, H and D in memory
};

// Most waves per workgroup with G groups of 4 nodes resident on each (FP64: 136
// registers for 4).
constexpr int units_waves(int G) { return G < 4 ? 4 : 12; }

struct DevUnits {
    DevResSync y;
    const int *tile_start;      // [ntiles + 1] first node (kernel order)
    const int *unit_start;      // [ntiles + 1] first unit
    const int *ustart;          // [ntiles + 1] offsets into ulist
    const int *ulist;           // distinct rows of each tile, kernel order, ascending
    const int *own_row;         // [ntiles] row number of the tile's first node
    const int *perm;            // kernel node -> node of the state buffer H
    const uint4 *prec;          // [units][64] row numbers, 8 x 16 bits
    int nsteps;
    int bytes;                  // of a state buffer
    int lds_rows;               // rows the LDS holds; FP64: the row after them is zero
    int lds_pos, lds_geo;       // units whose positions, geometry the LDS holds
};

// LDS bytes k_steps_units and k_steps_units32 need for a tile of `units` units
// and `rows` rows in a mode (units.h documents the pieces), with the counts
// they keep there; false when they do not fit.
bool units_plan64(SweUnits &u);
bool units_plan32(SweUnits &u);
// Kernel of a plan, its record packing and its launch.
void *units_kernel64(const SweUnits &u);
void *units_kernel32(const SweUnits &u);
bool units_plan_exact(SweUnits &u);
void *units_kernel_exact();
hipError_t units_launch_exact(swe_hip_ctx *c, int nsteps, const DevResSync &y);
void pack_weights64(swe_hip_ctx *c, int units);
int units_pack64(swe_hip_ctx *c, int units);
// The same for the ensemble stage kernel (k_ensemble.hip).
bool ensemble_plan(SweUnits &u);
int ensemble_rows(int halves);   // most rows of a tile
int ensemble_pack(swe_hip_ctx *c, int units);
int ensemble_prepare(swe_hip_ctx *c, std::string *err);
constexpr int kEnsNodes = 64;   // nodes per tile of the ensemble kernel with items of 8 members
int units_pack32(swe_hip_ctx *c, int units);
hipError_t units_launch64(swe_hip_ctx *c, int nsteps, const DevResSync &y);
hipError_t units_launch32(swe_hip_ctx *c, int nsteps, const DevResSync &y);
// The table part of a launch's arguments.
void units_tables(const swe_hip_ctx *c, int nsteps, const DevResSync &y, DevUnits *p);

// A 16-byte load of data no cache needs to keep.
template <typename T>
__device__ __forceinline__ T load_nt(const T *p)
{
    static_assert(sizeof(T) == 16, "16 bytes");
    return __builtin_bit_cast(T, __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p)));
}

}  // namespace swe
