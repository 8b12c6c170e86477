// dem_passes.h -- which force passes run and which wait for a rebuild, as the
// force kernel and the host (run_passes) both count it.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define DEM_PASSES_FN __host__ __device__ inline
#else
#define DEM_PASSES_FN inline
#endif

// The rebuild flag: the number of the first force pass that must not run on
// the present lists, doubled, plus one (so that it is never 0).
DEM_PASSES_FN uint32_t rebuild_at(uint32_t pass) { return pass << 1 | 1u; }

// Whether force pass `pass` has to wait for that rebuild.  A pass and the
// drift that it ends with, which asks for the next one, never confuse each
// other.
DEM_PASSES_FN bool waits_for_rebuild(uint32_t flag, uint32_t pass)
{
    return flag != 0 && (int32_t)(flag - rebuild_at(pass)) <= 0;
}

// How many of the passes launched so far, `pass` the last, wait for it.
DEM_PASSES_FN int64_t idle_passes(uint32_t flag, uint32_t pass)
{
    return waits_for_rebuild(flag, pass) ? (int32_t)(rebuild_at(pass) - flag) / 2 + 1 : 0;
}
