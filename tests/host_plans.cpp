// The launch plans of the kernels, which are plain host arithmetic, for the tests (host_plans.py).
#include "gs2d_direct_plan.hpp"

using namespace opscv;

extern "C" {

// tiles, channel runs; 0 where the tiled kernel is not taken
int direct_tiles(int elem, int64_t N, int64_t C, int64_t Hin, int64_t Win, int64_t Hout, int64_t Wout, int64_t* out)
{
    GridSamplerArgs a;
    a.elem = (Elem)elem;
    a.N = N;
    a.C = C;
    a.Hin = Hin;
    a.Win = Win;
    a.Hout = Hout;
    a.Wout = Wout;
    const DirectTilePlan p = direct_tile_plan(a);
    out[0] = p.tiles;
    out[1] = p.chan_runs;
    return p.ok ? 1 : 0;
}

}  // extern "C"
