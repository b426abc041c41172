// The autograd tape, device-resident: declared in include/paperkiln_amd.hpp (it is part of the
// library's C++ interface); this header adds the kernel launchers for the translation units that
// implement it.
#pragma once
#include "tensor.h"

namespace pk {
// The copies that products read of the current context's parameters, each with the parameter it follows.
struct ShadowCopy {
    const Variable* of;
    CastJob job;
};
std::vector<ShadowCopy> shadow_copies();
namespace ops {
// ops::embedding of rows already gathered, and ops::linear_cross_entropy as the root of a pass with its value to pinned host memory as well
Var embedding_of(const Var& table, const std::shared_ptr<Buffer>& ids, Tensor rows);
Var linear_cross_entropy_to(const Var& h, const Var& E, const std::shared_ptr<Buffer>& targets, int64_t chunk_rows, bool loss_is_root, float* pinned);
}  // namespace ops
}  // namespace pk
