// engines.hpp -- makers of the engines and batches, one source per precision
// (engine_*.hip), so that they compile side by side.
#pragma once
#include <memory>
#include "batch.hpp"
#include "engine.hpp"

namespace uaamg {

std::unique_ptr<EngineBase> make_engine_f64(int dim, const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s);
std::unique_ptr<EngineBase> make_engine_mixed_f64(int dim, const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s);
std::unique_ptr<EngineBase> make_engine_f32(int dim, const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s);
std::unique_ptr<EngineBase> make_engine_f32_2d(const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s);
// 3D; records_only: BF16 stencil records with FP32 level vectors
std::unique_ptr<EngineBase> make_engine_bf16(bool records_only, const uaamg_opts& o, const int n[3], const double h[3], const int wall[6], hipStream_t s);
std::unique_ptr<BatchBase> make_batch_f32(int dim, const uaamg_opts& o, hipStream_t s);
std::unique_ptr<BatchBase> make_batch_f32_2d(const uaamg_opts& o, hipStream_t s);
std::unique_ptr<BatchBase> make_batch_bf16(const uaamg_opts& o, hipStream_t s);

}  // namespace uaamg
