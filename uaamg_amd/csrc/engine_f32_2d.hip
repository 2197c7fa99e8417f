// engine_f32_2d.hip -- the 2D FP32 engine and batch.
#include "engine_impl.hpp"
#include "engines.hpp"

namespace uaamg {

std::unique_ptr<EngineBase> make_engine_f32_2d(const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s) {
    return std::make_unique<Engine<2, float, float>>(o, n, h, wall, s);
}
std::unique_ptr<BatchBase> make_batch_f32_2d(const uaamg_opts& o, hipStream_t s) {
    return std::make_unique<BatchEngine<2, float>>(o, s);
}

}  // namespace uaamg
