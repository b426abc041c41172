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
// ops::embedding of rows already gathered, and ops::linear_cross_entropy as the root of a pass with its value to pinned host memory as well, which
// writes E's gradient instead of adding to it where that has not been cleared (dE_unset)
Var embedding_of(const Var& table, const std::shared_ptr<Buffer>& ids, Tensor rows);
Var linear_cross_entropy_to(const Var& h, const Var& E, const std::shared_ptr<Buffer>& targets, int64_t chunk_rows, bool loss_is_root, float* pinned,
                            bool dE_unset = false);
// What a rotated projection's node and the attention that alone reads it share: the attention's backward turns dQ and dK back on their way out
// where its kernels do that, and the node then passes its gradient on as it is.
struct Turned {
    std::shared_ptr<Buffer> table;  // of k_rope_table
    int heads = 0;
    bool gradient_is_back = false;
};
// apply_rope(linear3(rmsnorm(x, norm_w), Wq, Wk, Wv), in place), the same three nodes, norm and rotation formed in the product where the
// kernels take them; the rotation from a table of k_rope_table for as many positions as a sequence has, where row r's position (pos) is r % seq_len
Var rms_linear3_rope(const Var& x, const Var& norm_w, const Var& Wq, const Var& Wk, const Var& Wv, const std::shared_ptr<Buffer>& pos, float theta, int head_dim, int rot_heads,
                     const std::shared_ptr<Buffer>& table, int64_t seq_len, std::shared_ptr<Turned>& turned);
// ops::attention_qkv of such a projection, which nothing else reads
Var attention_turned(const Var& qkv, const std::shared_ptr<Turned>& turned, int n_heads, float scale, int64_t seq_len, bool causal, int window, int sinks);
Var rms_gated_mlp(const Var& x, const Var& norm_w, const Var& gate, const Var& up, const Var& down, bool result_needed);  // gated_mlp(rmsnorm(x, norm_w), ..., x, ...)
}  // namespace ops
}  // namespace pk
