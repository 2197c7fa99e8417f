// engine_f32.hip -- the 3D FP32 engine and batch (and the choice by dimension).
#include "engine_impl.hpp"
#include "engines.hpp"

namespace uaamg {

std::unique_ptr<EngineBase> make_engine_f32(int dim, const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s) {
    if (dim == 2) return make_engine_f32_2d(o, n, h, wall, s);
    return std::make_unique<Engine<3, float, float>>(o, n, h, wall, s);
}
std::unique_ptr<BatchBase> make_batch_f32(int dim, const uaamg_opts& o, hipStream_t s) {
    if (dim == 2) return make_batch_f32_2d(o, s);
    return std::make_unique<BatchEngine<3, float>>(o, s);
}

}  // namespace uaamg
