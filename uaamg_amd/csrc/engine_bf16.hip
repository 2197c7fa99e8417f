// engine_bf16.hip -- the 3D engines with BF16 coarse levels or BF16 records, and the batch.
#include "engine_impl.hpp"
#include "engines.hpp"

namespace uaamg {

std::unique_ptr<EngineBase> make_engine_bf16(bool records_only, const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s) {
    if (records_only) return std::make_unique<Engine<3, float, float, __bf16>>(o, n, h, wall, s);
    return std::make_unique<Engine<3, float, __bf16>>(o, n, h, wall, s);
}
std::unique_ptr<BatchBase> make_batch_bf16(const uaamg_opts& o, hipStream_t s) {
    return std::make_unique<BatchEngine<3, __bf16>>(o, s);
}

}  // namespace uaamg
