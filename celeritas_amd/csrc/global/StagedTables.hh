//----------------------------------*-C++-*----------------------------------//
// celeritas_amd: MI355X-native per-step transport loop
//---------------------------------------------------------------------------//
//! \file global/StagedTables.hh
//! LDS staging of the physics and geometry tables a step kernel reads per
//! track.
//!
//! The particle and process records, grid headers and grid values, and the
//! material, MSC and fluctuation records live in one contiguous device
//! region (PhysicsParamsRef::hot_base, hot_bytes), and so do the surface,
//! face, volume logic, bounding box and connectivity tables of the geometry
//! (GeoParamsRef::hot_base, hot_bytes). A kernel launched with enough
//! dynamic LDS copies the regions it reads once per workgroup and continues
//! with a params view whose table pointers are rebased into LDS, so the
//! chains of dependent table reads of a track (particle -> process -> grid
//! header -> values; volume -> faces) are served from LDS instead of L2. The
//! data are the same bytes, so results are bit-identical to the unstaged
//! path. StagingRules.hh says which regions a launch stages.
//---------------------------------------------------------------------------//
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "corecel/WaveOps.hh"
#include "CoreData.hh"
#include "StagingRules.hh"
#include "StepExecutors.hh"

namespace celeritas_amd
{
//---------------------------------------------------------------------------//
/*!
 * Whether any thread of this workgroup maps to a slot.
 *
 * A sorted launch covers all slots but its range is read on the device, so
 * most of its workgroups can be empty: they return before staging (the
 * answer is uniform over the workgroup, so no barrier is left waiting).
 */
__device__ __forceinline__ bool workgroup_has_work(ThreadSlots const& ts,
                                                   size_type size)
{
    size_type const first = blockIdx.x * blockDim.x;
    if (ts.range)
    {
        size_type const end = ts.range_end ? *ts.range_end : ts.range[1];
        return first < end - ts.range[0];
    }
    return first < size;
}

namespace detail
{
template<class T>
__device__ __forceinline__ T const* rebase(T const* p, char const* from, char* to)
{
    return p ? reinterpret_cast<T const*>(to + (reinterpret_cast<char const*>(p) - from))
             : p;
}

/*!
 * Copy a 16-byte-aligned region into LDS (no barrier).
 *
 * Each thread has a batch of loads in flight before it writes any: a loop
 * of load and write waited for the memory once per 4 KiB, 12 times for the
 * 46 KB of the charged along-step (2^20 slots: pre-step 67 -> 61 us a step;
 * full TestEm3 transport 885 -> 874 ms).
 */
__device__ __forceinline__ void copy_region(char const* from, unsigned int n, char* to)
{
    constexpr unsigned int batch = 8;
    auto const* src = reinterpret_cast<uint4 const*>(from);
    auto* dst = reinterpret_cast<uint4*>(to);
    unsigned int const count = n / 16;
    for (unsigned int first = threadIdx.x; first < count; first += batch * blockDim.x)
    {
        // Beyond the end the last word again: without a condition on the
        // writes the loads stay together
        uint4 v[batch];
#pragma unroll
        for (unsigned int u = 0; u < batch; ++u)
            v[u] = src[min(first + u * blockDim.x, count - 1)];
#pragma unroll
        for (unsigned int u = 0; u < batch; ++u)
            dst[min(first + u * blockDim.x, count - 1)] = v[u];
    }
}

//! Physics table pointers rebased into LDS
__device__ __forceinline__ void rebase_physics(PhysicsParamsRef* r, char* to)
{
    PhysicsParamsRef const pp = *r;
    char const* from = pp.hot_base;
    r->particle = rebase(pp.particle, from, to);
    r->grids = rebase(pp.grids, from, to);
    r->grid_reals = rebase(pp.grid_reals, from, to);
    r->mass = rebase(pp.mass, from, to);
    r->charge = rebase(pp.charge, from, to);
    r->materials = rebase(pp.materials, from, to);
    r->msc_material = rebase(pp.msc_material, from, to);
    r->msc_par_mat = rebase(pp.msc_par_mat, from, to);
    r->fluct = rebase(pp.fluct, from, to);
    r->model_class = rebase(pp.model_class, from, to);
}

//! Pointers of the tables that finding distances reads
__device__ __forceinline__ void rebase_geometry(GeoParamsRef* r, char* to)
{
    GeoParamsRef const g = *r;
    char const* from = g.hot_base;
    r->surfaces = rebase(g.surfaces, from, to);
    r->planes = rebase(g.planes, from, to);
    r->volumes = rebase(g.volumes, from, to);
    r->faces = rebase(g.faces, from, to);
    r->logic = rebase(g.logic, from, to);
}

//! Pointers of the tables that only boundary crossings read
__device__ __forceinline__ void rebase_crossing(GeoParamsRef* r, char* to)
{
    GeoParamsRef const g = *r;
    char const* from = g.hot_base;
    r->vol_bbox = rebase(g.vol_bbox, from, to);
    r->conn_begin = rebase(g.conn_begin, from, to);
    r->conn_size = rebase(g.conn_size, from, to);
    r->conn_vols = rebase(g.conn_vols, from, to);
}
}  // namespace detail

/*!
 * Stage the tables a launch reads per track into its dynamic LDS and
 * return the params with those tables' pointers in LDS (the physics region
 * first, then the geometry region).
 *
 * Every thread of the workgroup must call this before any of them returns
 * (it contains a workgroup barrier). The launcher gives the kernel the LDS
 * its staging needs (StagingRules.hh) and instantiates it with that staging
 * only when the regions fit: the table pointers then derive from the LDS
 * array alone, so the compiler reads them with LDS instructions and 32-bit
 * addresses.
 */
template<Staging S>
__device__ __forceinline__ CoreParamsRef stage(CoreParamsRef const& params, void* lds)
{
    if constexpr (S == Staging::none)
    {
        return params;
    }
    else
    {
        CoreParamsRef r = params;
        char* to = static_cast<char*>(lds);
        unsigned int offset = 0;
        if constexpr (S == Staging::physics || S == Staging::both)
        {
            detail::copy_region(params.phys.hot_base, params.phys.hot_bytes, to);
            detail::rebase_physics(&r.phys, to);
            offset = params.phys.hot_bytes;
        }
        if constexpr (S == Staging::geometry || S == Staging::both)
        {
            detail::copy_region(params.geo.hot_base, params.geo.track_bytes, to + offset);
            detail::rebase_geometry(&r.geo, to + offset);
        }
        if constexpr (S == Staging::crossing)
        {
            detail::copy_region(params.geo.hot_base, params.geo.hot_bytes, to);
            detail::rebase_geometry(&r.geo, to);
            detail::rebase_crossing(&r.geo, to);
        }
        __syncthreads();
        return r;
    }
}

//! Stage the physics tables when \c Staged (see stage)
template<bool Staged>
__device__ __forceinline__ CoreParamsRef stage_tables(CoreParamsRef const& params,
                                                      void* lds)
{
    return stage<Staged ? Staging::physics : Staging::none>(params, lds);
}

//---------------------------------------------------------------------------//
}  // namespace celeritas_amd
