// engine_f64.hip -- the FP64 engines.
#include "engine_impl.hpp"
#include "engines.hpp"

namespace uaamg {

std::unique_ptr<EngineBase> make_engine_f64(int dim, const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s) {
    if (dim == 2) return std::make_unique<Engine<2, double, double>>(o, n, h, wall, s);
    return std::make_unique<Engine<3, double, double>>(o, n, h, wall, s);
}

}  // namespace uaamg
