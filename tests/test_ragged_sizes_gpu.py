"""GPU tests at the sizes where the kernels' edges lie: token counts, vocabularies, head sizes and sequence lengths that
are no multiple of a tile, a chunk or a wavefront."""
import numpy as np
import pytest
import torch

from paperkiln_amd import blockops, synth
from paperkiln_amd.llama import Llama

pytestmark = pytest.mark.gpu


def rel(a, b):
    return max(float(np.linalg.norm(a[k].astype(np.float64) - b[k]) / max(np.linalg.norm(b[k].astype(np.float64)), 1e-30)) for k in b)


@pytest.mark.parametrize("tokens,seq", [(2051, 293), (2052, 0), (77, 11)])
def test_bf16_training_on_a_ragged_token_count(tokens, seq):
    """Weight gradients contract over the tokens; where those are the row index of both operands the library's own
    GEMM takes any number of them (held back and grouped from 2048 on). Against the library GEMM, same operands."""
    m = Llama(vocab=504, d=512, n_layers=1, n_heads=8, d_ff=1376, compute_dtype="bf16", seed=8)
    toks = synth.randint(3, tokens + 1, 504)
    before = blockops.set_gemm_backend(0)
    try:
        want_loss, _ = m.loss_backward(toks[:-1], toks[1:], seq)
        want = m.grads()
        blockops.set_gemm_backend(1)
        for ck in (False, True):
            loss, _ = m.loss_backward(toks[:-1], toks[1:], seq, checkpoint=ck)
            assert abs(loss - want_loss) < 1e-3
            assert rel(m.grads(), want) < 2e-2
    finally:
        blockops.set_gemm_backend(before)
        m.close()
