//----------------------------------*-C++-*----------------------------------//
// celeritas_amd: MI355X-native per-step transport loop
//---------------------------------------------------------------------------//
//! \file global/StagingRules.hh
//! Which of its tables a step kernel copies into LDS.
//!
//! Copying costs a workgroup its share of the CU's LDS, so a region is staged
//! while it leaves the kernel the workgroups that it needs; above that the
//! kernel reads the tables in place. The lines below come from TestEm3
//! transports (10,000 primaries, 2^20 slots, 256-thread workgroups) with 50
//! to 110 layers and 7 to 10 grid points a decade, each kernel timed alone.
//---------------------------------------------------------------------------//
#pragma once

#include "CoreData.hh"

namespace celeritas_amd
{
//---------------------------------------------------------------------------//
//! LDS of a CU and the unit that it is handed out in [B]
inline constexpr unsigned int lds_per_cu = 160 * 1024;
inline constexpr unsigned int lds_unit = 1280;

//! Largest LDS of a workgroup of which so many fit a CU
constexpr unsigned int lds_share(unsigned int workgroups)
{
    return lds_per_cu / workgroups / lds_unit * lds_unit;
}

/*!
 * Physics tables, and those that finding distances reads, alone or together:
 * three workgroups.
 *
 * That is what the registers of the charged along-step and the interactions
 * allow. Staging both regions takes the charged along-step from 173 to 164
 * us a step at 53,296 B, and from 170 to 197 us at 55,648 B, where a third
 * workgroup no longer fits. The pre-step and the neutral along-step have
 * registers for five, but three with their tables at hand are faster than
 * five without: 80 -> 73 us (49,456 B), 52.7 -> 51.4 us (43,968 B).
 */
inline constexpr unsigned int max_staged_tables = lds_share(3);

/*!
 * All geometry tables: four workgroups.
 *
 * The boundary kernel has registers for eight and little work, so it gains
 * less and stops earlier: 25.5 -> 24.4 us at 39,760 B, 25.4 -> 26.4 us at
 * 48,592 B.
 */
inline constexpr unsigned int max_staged_crossing = lds_share(4);

//---------------------------------------------------------------------------//
//! Dynamic LDS bytes of a launch staging the physics tables (0: the tables
//! stay in HBM)
inline unsigned int staged_table_bytes(CoreParamsRef const& p)
{
    unsigned int const n = p.phys.hot_bytes;
    return n <= max_staged_tables ? n : 0;
}

//! Dynamic LDS bytes of a launch staging the tables that finding distances
//! reads
inline unsigned int staged_geo_bytes(CoreParamsRef const& p)
{
    unsigned int const n = p.geo.track_bytes;
    return n <= max_staged_tables ? n : 0;
}

//! Dynamic LDS bytes of a launch staging all geometry tables
inline unsigned int staged_crossing_bytes(CoreParamsRef const& p)
{
    unsigned int const n = p.geo.hot_bytes;
    return n <= max_staged_crossing ? n : 0;
}

//! Dynamic LDS bytes of a launch staging physics and distances (physics first)
inline unsigned int staged_both_bytes(CoreParamsRef const& p)
{
    unsigned int const a = staged_table_bytes(p);
    unsigned int const b = staged_geo_bytes(p);
    return (a > 0 && b > 0 && a + b <= max_staged_tables) ? a + b : 0;
}

//---------------------------------------------------------------------------//
//! What a launch stages in LDS
enum class Staging
{
    none,
    physics,
    geometry,  //!< what finding distances reads
    crossing,  //!< all of the geometry
    both,  //!< physics and geometry
};

//! What the charged along-step stages
inline Staging charged_staging(CoreParamsRef const& p)
{
    return staged_both_bytes(p)    ? Staging::both
           : staged_table_bytes(p) ? Staging::physics
                                   : Staging::none;
}

//---------------------------------------------------------------------------//
}  // namespace celeritas_amd
