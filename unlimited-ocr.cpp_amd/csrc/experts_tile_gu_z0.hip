// INT4 grouped expert GEMM, 64- and 128-slot tiles: gate/up pass, without zero offsets
// (one of the four translation units of experts_tile.hpp's kernels, compiled in parallel).
#include "experts_tile.hpp"

namespace uocr_hip {

hipError_t launch_tile_gu_z0(const ExpertArgs& a, int max_tiles, hipStream_t st) {
    return launch_int4_tile<true, false>(a, max_tiles, st);
}

}  // namespace uocr_hip
