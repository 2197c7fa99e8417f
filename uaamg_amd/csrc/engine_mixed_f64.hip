// engine_mixed_f64.hip -- the engines with FP64 vectors and FP32 coarse levels.
#include "engine_impl.hpp"
#include "engines.hpp"

namespace uaamg {

std::unique_ptr<EngineBase> make_engine_mixed_f64(int dim, const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s) {
    if (dim == 2) return std::make_unique<Engine<2, double, float>>(o, n, h, wall, s);
    return std::make_unique<Engine<3, double, float>>(o, n, h, wall, s);
}

}  // namespace uaamg
