// relax_push_lds.hip -- the relaxation kernel variants for batches of push queries only whose boundary
// candidates are gathered in LDS first (boundary_mode 0).
#include "relax_kernels.hpp"

#include "bfn_launch.hpp"

namespace bfn {

hipError_t relax_launch_push_lds(std::uint32_t block, bool persistent, bool cooperative,
                        std::uint32_t grid, std::size_t lds_bytes, std::uint32_t max_v,
                        std::uint32_t work_words, const DevGraph& g, const DevBatch& b,
                        hipStream_t stream) {
  return relax_launch_engines<kEnginesPushLds>(block, persistent, cooperative, grid, lds_bytes, max_v,
                                   work_words, g, b, stream);
}

hipError_t relax_occupancy_push_lds(std::uint32_t block, bool persistent, bool instrumented,
                           std::uint32_t min_waves, std::size_t lds_bytes, int* blocks_per_cu) {
  return relax_occupancy_engines<kEnginesPushLds>(block, persistent, instrumented, min_waves, lds_bytes,
                                      blocks_per_cu);
}

}  // namespace bfn
