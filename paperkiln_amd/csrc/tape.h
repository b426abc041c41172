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
// apply_rope(linear3(x, Wq, Wk, Wv), in place), the same two nodes, the rotation formed in the product where the kernels take it: from a
// table of k_rope_table for as many positions as a sequence has, where row r's position (pos) is r % seq_len
Var linear3_rope(const Var& x, const Var& Wq, const Var& Wk, const Var& Wv, const std::shared_ptr<Buffer>& pos, float theta, int head_dim, int rot_heads,
                 const std::shared_ptr<Buffer>& table, int64_t seq_len);
}  // namespace ops
}  // namespace pk
