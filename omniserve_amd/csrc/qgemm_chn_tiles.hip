// The per-channel products of prompts in 256 x 256 tiles (qgemm_group_tiles.h).  A file of its own: see qgemm_silu_rows.hip.
#include "qgemm_kernel.h"
#include "qgemm_group_tiles.h"
using namespace omni;

void omni::launch_chn_tiles(const GemmArgs& a, const TileShare& share, hipStream_t st) { launch_w4_tiles_as<MODE_CHN, false>(a, share, st); }
