// Prefill expert GEMM: the host-side dispatch. The kernels and their
// template launchers live in experts_prefill.hpp (256-slot tiles) and
// experts_tile.hpp (64 and 128); their instantiations are split over four
// translation units each (gate/up or down, with or without zero offsets) so
// that they compile in parallel.
#include "experts_prefill.hpp"

namespace uocr_hip {

hipError_t launch_prefill_gu_z0(const ExpertArgs& a, int max_tiles, hipStream_t st);
hipError_t launch_prefill_gu_z1(const ExpertArgs& a, int max_tiles, hipStream_t st);
hipError_t launch_prefill_dn_z0(const ExpertArgs& a, int max_tiles, hipStream_t st);
hipError_t launch_prefill_dn_z1(const ExpertArgs& a, int max_tiles, hipStream_t st);

hipError_t launch_tile_gu_z0(const ExpertArgs& a, int max_tiles, hipStream_t st);
hipError_t launch_tile_gu_z1(const ExpertArgs& a, int max_tiles, hipStream_t st);
hipError_t launch_tile_dn_z0(const ExpertArgs& a, int max_tiles, hipStream_t st);
hipError_t launch_tile_dn_z1(const ExpertArgs& a, int max_tiles, hipStream_t st);

hipError_t launch_experts_prefill(const ExpertArgs& a, bool gate_up, int max_tiles, hipStream_t st) {
    if (max_tiles <= 0) return hipSuccess;
    if (a.bm != kPrefillBigTileRows) {
        if (a.z0) return gate_up ? launch_tile_gu_z1(a, max_tiles, st) : launch_tile_dn_z1(a, max_tiles, st);
        return gate_up ? launch_tile_gu_z0(a, max_tiles, st) : launch_tile_dn_z0(a, max_tiles, st);
    }
    if (a.z0) return gate_up ? launch_prefill_gu_z1(a, max_tiles, st) : launch_prefill_dn_z1(a, max_tiles, st);
    return gate_up ? launch_prefill_gu_z0(a, max_tiles, st) : launch_prefill_dn_z0(a, max_tiles, st);
}

}  // namespace uocr_hip
