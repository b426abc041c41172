"""GPU tests at the sizes where the kernels' edges lie: token counts, vocabularies, head sizes and sequence lengths that
are no multiple of a tile, a chunk or a wavefront."""
import ctypes

import numpy as np
import pytest
import torch

from paperkiln_amd import _lib, blockops, ops, synth
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


@pytest.mark.parametrize("vocab,d,ff,layers,tokens,seq", [(301, 64, 176, 2, 77, 11), (1001, 128, 344, 1, 693, 77),
                                                          (12345, 256, 688, 1, 2600, 650), (17, 64, 176, 1, 64, 0),
                                                          (3122, 512, 1368, 1, 2924, 34), (20001, 512, 1368, 1, 4100, 820)])
def test_bf16_training_with_any_vocabulary(vocab, d, ff, layers, tokens, seq):
    """The tied head's cross-entropy inside its product, with a vocabulary padded to a multiple of 8 (small and large
    tiles, several rounds of each), and the weight gradients of few tokens in one launch. Against the library GEMM, same operands."""
    m = Llama(vocab=vocab, d=d, n_layers=layers, n_heads=d // 32, d_ff=ff, compute_dtype="bf16", seed=8)
    toks = synth.randint(3, tokens + 1, vocab)
    toks[:4] = vocab - 1  # the last word is used, as input and as target
    before = blockops.set_gemm_backend(0)
    try:
        want_loss, _ = m.loss_backward(toks[:-1], toks[1:], seq)
        want = m.grads()
        blockops.set_gemm_backend(1)
        for ck in (False, True):
            loss, _ = m.loss_backward(toks[:-1], toks[1:], seq, checkpoint=ck)
            assert abs(loss - want_loss) < 1e-3
            assert rel(m.grads(), want) < 2e-2
        assert m.loss_backward(toks[:-1], toks[1:], seq, backward=False)[0] == loss
        m.adamw_step(1e-3)  # the padded copy is refreshed in place
        a, _ = m.loss_backward(toks[:-1], toks[1:], seq)
        blockops.set_gemm_backend(0)
        assert abs(a - m.loss_backward(toks[:-1], toks[1:], seq)[0]) < 1e-3
    finally:
        blockops.set_gemm_backend(before)
        m.close()


@pytest.mark.parametrize("d,ff,tokens,seq", [(64, 40, 33, 11), (96, 200, 1300, 130), (256, 1000, 2050, 410), (512, 1368, 700, 350),
                                             (64, 4104, 8200, 820), (800, 304, 8200, 820)])
def test_bf16_gated_product_in_its_projections(d, ff, tokens, seq):
    """SwiGLU in the gate|up projection and in the down projection's dX, with and without gate and up being kept, against the passes
    of their own beside the library's products: the kernel of few tiles, 128 x 128 and 256 x 256 tiles, a d_ff that ends inside
    one, and a contraction (800) too long for the form, which takes those passes."""
    test_bf16_training_with_any_vocabulary(130, d, ff, 1, tokens, seq)


@pytest.mark.parametrize("d,ff,tokens,seq", [(192, 512, 5940, 135), (128, 344, 6754, 614), (96, 200, 3001, 3001), (64, 176, 16380, 819), (64, 40, 1024, 128)])
def test_bf16_weight_gradients_in_slices(d, ff, tokens, seq):
    """A narrow block's weight gradients over many tokens: one launch whose contraction is cut, the last slice shorter, and its sum; the
    last case has too few tokens for two slices of 512 to pay."""
    test_bf16_training_with_any_vocabulary(130, d, ff, 2, tokens, seq)


@pytest.mark.parametrize("d,ff,tokens,seq", [(64, 20, 33, 11), (64, 344, 2100, 420), (256, 250, 400, 100), (288, 256, 800, 100), (128, 90, 500, 100)])
def test_fp32_gated_product_in_its_projections(d, ff, tokens, seq):
    """The same in fp32, with each of its tiles."""
    test_fp32_training_on_ragged_sizes(130, d, ff, tokens, seq)


@pytest.mark.parametrize("all_heads", [False, True])
@pytest.mark.parametrize("dtype,d,heads,tokens,seq", [
    ("fp32", 64, 2, 33, 11), ("fp32", 96, 3, 77, 0), ("fp32", 128, 4, 516, 129), ("fp32", 192, 3, 300, 30), ("fp32", 256, 4, 1025, 205),
    ("fp32", 24, 2, 70, 7), ("bf16", 64, 2, 33, 11), ("bf16", 128, 4, 516, 129), ("bf16", 24, 2, 70, 7), ("bf16", 256, 4, 2050, 410),
    ("bf16", 320, 5, 2112, 33), ("bf16", 512, 8, 2048, 128), ("bf16", 512, 16, 1400, 100), ("bf16", 384, 3, 3001, 3001),
    ("fp32", 40, 5, 50, 10), ("fp32", 512, 8, 100, 25), ("fp32", 448, 7, 17, 17), ("fp32", 100, 5, 1100, 55), ("fp32", 128, 2, 1700, 85),
    ("bf16", 40, 5, 50, 10), ("bf16", 100, 5, 1100, 55), ("bf16", 512, 8, 17, 17), ("bf16", 68, 1, 200, 40)])
def test_norm_and_rope_in_the_projection(dtype, d, heads, tokens, seq, all_heads):
    """Rows normalised where the q|k|v and gate|up products load them, kept and not kept, and q and k turned on their way out, from a table,
    against the passes of their own beside the library's products: tiles of 16 to 128 rows of sequences shorter and longer than one, thirds
    that end inside a tile, widths below a chunk of the contraction, beside one and past what a workgroup holds of it at once, head sizes that
    are no multiple of 8, and a second pass with longer sequences than the table has."""
    m = Llama(vocab=130, d=d, n_layers=1, n_heads=heads, d_ff=2 * d, compute_dtype=dtype, rope_all_heads=all_heads, seed=8)
    toks = synth.randint(3, tokens + 1, 130)
    tol = 1e-5 if dtype == "fp32" else 2e-2
    before = blockops.set_gemm_backend(0)
    try:
        for sl in (seq, tokens):
            blockops.set_gemm_backend(0)
            want_loss, _ = m.loss_backward(toks[:-1], toks[1:], sl)
            want = m.grads()
            blockops.set_gemm_backend(1)
            for ck in (False, True):
                loss, _ = m.loss_backward(toks[:-1], toks[1:], sl, checkpoint=ck)
                assert abs(loss - want_loss) < (1e-5 if dtype == "fp32" else 1e-3)
                assert rel(m.grads(), want) < tol
    finally:
        blockops.set_gemm_backend(before)
        m.close()


@pytest.mark.parametrize("all_heads", [False, True])
@pytest.mark.parametrize("dtype,d,heads,tokens,seq", [
    ("fp32", 64, 2, 33, 11), ("fp32", 40, 5, 50, 10), ("fp32", 192, 2, 1030, 515), ("fp32", 256, 2, 1538, 769), ("bf16", 64, 2, 33, 11),
    ("bf16", 80, 1, 70, 35), ("bf16", 96, 1, 700, 350), ("bf16", 192, 2, 1030, 515), ("bf16", 512, 8, 4084, 1021), ("bf16", 768, 8, 4000, 500)])
def test_rope_undone_in_attention_backward(dtype, d, heads, tokens, seq, all_heads):
    """dQ and dK turned back where the attention kernels write them against a pass of its own, which a window with sinks has: a window of all
    keys but the first and one sink see what causal attention sees. Where bf16 gradients are rounded differs: P, dS, dQ or dK and the turned
    ones, 2 ^ -9 each of a norm."""
    toks = synth.randint(3, tokens + 1, 130)
    got = []
    for window, sinks in ((seq - 1, 1), (0, 0)):
        m = Llama(vocab=130, d=d, n_layers=1, n_heads=heads, d_ff=2 * d, compute_dtype=dtype, rope_all_heads=all_heads, window=window, sinks=sinks, seed=8)
        got.append((m.loss_backward(toks[:-1], toks[1:], seq)[0], m.grads()))
        m.close()
    assert abs(got[0][0] - got[1][0]) < (1e-5 if dtype == "fp32" else 1e-3)
    assert rel(got[1][1], got[0][1]) < (1e-5 if dtype == "fp32" else 4 * 2.0 ** -9)


def exact_block_model(params, toks, seq, heads, rot_heads, window):
    """Loss and gradients in float64 of a Llama of one block (llama.cpp:25-89) whose attention sees the last `window` keys."""
    P = {k: torch.from_numpy(v).cuda().double().requires_grad_() for k, v in params.items()}
    W = {k.split(".")[-2]: v for k, v in P.items()}
    x, y = (torch.from_numpy(t.astype(np.int64)).cuda() for t in (toks[:-1], toks[1:]))
    E = W["embed_tokens"]
    n, d = len(x), E.shape[1]
    dk = d // heads
    norm = lambda t, w: t * w.reshape(1, -1) / torch.sqrt((t * t).mean(1, keepdim=True) + 1e-5)  # noqa: E731
    angle = (torch.arange(n, device="cuda") % seq)[:, None] / 10000.0 ** (torch.arange(0, dk, 2, device="cuda").double() / dk)
    c, s = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def turn(t):  # [n, heads, dk], the first rot_heads of them
        a, b = t[:, :rot_heads, 0::2], t[:, :rot_heads, 1::2]
        return torch.cat([torch.stack([a * c - b * s, a * s + b * c], -1).reshape(n, rot_heads, dk), t[:, rot_heads:]], 1)

    h = E[x]
    u = norm(h, W["input_layernorm"])
    q, k, v = ((u @ W[w]).reshape(n, heads, dk) for w in ("q_proj", "k_proj", "v_proj"))
    q, k, v = (t.reshape(-1, seq, heads, dk).transpose(1, 2).contiguous() for t in (turn(q), turn(k), v))
    i, j = torch.arange(seq, device="cuda")[:, None], torch.arange(seq, device="cuda")[None, :]
    scores = (q @ k.transpose(2, 3).contiguous() / dk ** 0.5).masked_fill((j > i) | (j + window <= i), float("-inf"))
    h = h + (torch.softmax(scores, -1) @ v).transpose(1, 2).reshape(n, d) @ W["o_proj"]
    u = norm(h, W["post_attention_layernorm"])
    h = h + (torch.nn.functional.silu(u @ W["gate_proj"]) * (u @ W["up_proj"])) @ W["down_proj"]
    loss = torch.nn.functional.cross_entropy(norm(h, W["norm"]) @ E.T, y)
    loss.backward()
    return float(loss), {k: t.grad.cpu().numpy() for k, t in P.items()}


@pytest.mark.parametrize("all_heads", [False, True])
@pytest.mark.parametrize("dtype,d,heads,tokens,seq,window,form", [
    ("fp32", 64, 2, 33, 11, 4, "F32_SPLIT"), ("fp32", 96, 1, 700, 350, 64, "F32_SPLIT"), ("fp32", 256, 2, 1538, 769, 200, "F32_PARTS_ALL"),
    ("fp32", 512, 8, 4084, 1021, 128, "F32_PARTS"), ("bf16", 64, 2, 33, 11, 4, "SPLIT"), ("bf16", 80, 1, 70, 35, 9, "SPLIT"),
    ("bf16", 128, 2, 2000, 250, 30, "SPLIT"), ("bf16", 256, 2, 1538, 769, 200, "SPLIT"), ("bf16", 512, 8, 4084, 1021, 128, "SPLIT_JOINED"),
    ("bf16", 768, 8, 4000, 500, 100, "SPLIT_JOINED")])
def test_rope_undone_under_a_band(dtype, d, heads, tokens, seq, window, form, all_heads):
    """dQ and dK turned back where the attention kernels write them, under a band without sinks, against float64. bf16: some twenty tensors of a pass are
    rounded, each by 2 ^ -9 of a norm at most; fp32: a chain of sums of up to 4084 terms, sqrt(4084) 2 ^ -24 = 4e-6 each."""
    assert bwd_form((tokens // seq, seq, heads, heads, 1, window, 0), d // heads, torch.float32 if dtype == "fp32" else torch.bfloat16) == form
    m = Llama(vocab=130, d=d, n_layers=1, n_heads=heads, d_ff=2 * d, compute_dtype=dtype, rope_all_heads=all_heads, window=window, seed=8)
    toks = synth.randint(3, tokens + 1, 130)
    loss, _ = m.loss_backward(toks[:-1], toks[1:], seq)
    want_loss, want = exact_block_model(m.params(), toks, seq, heads, heads if all_heads else 1, window)
    assert abs(loss - want_loss) < (1e-5 if dtype == "fp32" else 1e-3)
    got = m.grads()
    assert rel(got, {k: g.reshape(got[k].shape) for k, g in want.items()}) < (2e-5 if dtype == "fp32" else 20 * 2.0 ** -9)
    m.close()


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_rope_table_of_passes_on_several_streams(dtype):
    """The table of cosines and sines grows with the longest sequence yet, on whichever stream that pass runs, and serves shorter ones behind it on others: the
    bits of models that have had no other pass."""
    cfg = dict(vocab=130, d=64, n_layers=1, n_heads=2, d_ff=128, compute_dtype=dtype, rope_all_heads=True, seed=8)
    toks = synth.randint(3, 321, 130)
    m, streams = Llama(**cfg), [torch.cuda.Stream() for _ in range(3)]
    for i, seq in enumerate((16, 64, 32, 320, 160, 80)):
        got = m.loss_backward(toks[:320], toks[1:], seq, stream=streams[i % 3].cuda_stream)[0], m.grads()
        fresh = Llama(**cfg)
        assert fresh.loss_backward(toks[:320], toks[1:], seq)[0] == got[0]
        assert all(np.array_equal(g, got[1][k]) for k, g in fresh.grads().items())
        fresh.close()
    m.close()


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("vocab,d,ff,layers", [(130, 64, 176, 8), (37, 12, 20, 1), (37, 6, 10, 1)])
def test_optimiser_step_writes_the_copies(vocab, d, ff, layers, dtype):
    """AdamW with the products' copies of the parameters written in the same pass: more parameters than one launch takes, sizes
    that are no multiple of 8, and of 4 (two passes). Against float64; and a model made from the result has the same loss.
    An update's terms are each within their rounding of 1: 1e-5 of the rate, and the sum's own."""
    m = Llama(vocab=vocab, d=d, n_layers=layers, n_heads=1, d_ff=ff, compute_dtype=dtype, seed=8)
    toks = synth.randint(3, 65, vocab)
    m1 = {k: np.zeros(v.shape) for k, v in m.params().items()}
    m2 = {k: np.zeros(v.shape) for k, v in m1.items()}
    for t in (1, 2):
        m.loss_backward(toks[:-1], toks[1:], 32)
        g, p = m.grads(), m.params()
        norm = m.adamw_step(1e-2, max_norm=0.5)
        for k, now in m.params().items():
            gk = g[k].astype(np.float64) * min(1.0, 0.5 / norm)
            m1[k], m2[k] = 0.9 * m1[k] + 0.1 * gk, 0.999 * m2[k] + 0.001 * gk * gk
            step = m1[k] / (1 - 0.9 ** t) / (np.sqrt(m2[k] / (1 - 0.999 ** t)) + 1e-8) + 0.01 * p[k]
            assert (np.abs(now - (p[k] - 1e-2 * step)) <= 1e-2 * 1e-5 + 2e-7 * np.abs(now)).all(), (k, t)
    fresh = Llama(vocab=vocab, d=d, n_layers=layers, n_heads=1, d_ff=ff, compute_dtype=dtype, seed=9)
    fresh.set_params(m.params())
    assert fresh.loss_backward(toks[:-1], toks[1:], 32)[0] == m.loss_backward(toks[:-1], toks[1:], 32)[0]
    m.close()
    fresh.close()


@pytest.mark.parametrize("dtype,tol", [("fp32", 1e-5), ("bf16", 1e-2)])
@pytest.mark.parametrize("vocab", [512, 4000])
def test_first_and_last_launch_of_a_pass(vocab, dtype, tol):
    """2048 tokens of 256 columns are gathered in the launch that begins a pass, 2064 are not; 0.4 M parameters form the clip's factor in
    the optimiser's workgroups, 1.3 M in a launch before. A batch is the mean of its parts (another order of sums; in bf16 dlogits
    rounded at another scale, 2^-9 of each), the norm that of the gradients read back."""
    m = Llama(vocab=vocab, d=256, n_layers=1, n_heads=4, d_ff=64, compute_dtype=dtype, seed=5)
    toks = synth.randint(11, 2065, vocab)
    parts = [(0, 2048), (2048, 2064)]
    loss, grads = 0.0, None
    for lo, hi in parts:
        w = (hi - lo) / 2064
        one = m.loss_backward(toks[lo:hi], toks[lo + 1:hi + 1], 16)[0]
        loss, g = loss + w * one, m.grads()
        grads = {k: w * g[k].astype(np.float64) + (grads[k] if grads else 0.0) for k in g}
    whole = m.loss_backward(toks[:2064], toks[1:2065], 16)[0]
    assert abs(whole - loss) < 1e-5 * loss
    g = m.grads()
    assert rel(g, grads) < tol
    norm = m.adamw_step(1e-3, max_norm=1e-3)
    assert abs(norm - np.sqrt(sum((x.astype(np.float64) ** 2).sum() for x in g.values()))) < 1e-6 * norm
    assert rel({k: x * (norm / 1e-3) for k, x in m.grads().items()}, g) < 1e-6  # scaled where they lie
    m.close()


def exact_attention(q, k, v, d_o, scale, causal, window, sinks, given_o=None):
    """O, LSE, dQ, dK, dV in float64 (src/ops.cpp:863-1027) of [B,T,H,dk] tensors, K / V heads shared by groups. given_o: the O
    whose rowsum(dO .* O) the gradients are formed with, as a backward is given it; the exact O otherwise."""
    q, k, v, d_o = (x.double().permute(0, 2, 1, 3).contiguous() for x in (q, k, v, d_o))
    B, Hq, T, dk = q.shape
    rep = Hq // k.shape[1]
    kx, vx = (x.repeat_interleave(rep, 1) for x in (k, v))
    i, j = torch.arange(T, device=q.device)[:, None], torch.arange(T, device=q.device)[None, :]
    vis = (j <= i) if causal else torch.ones(T, T, dtype=torch.bool, device=q.device)
    if window > 0:
        vis = vis & ((j + window > i) | (j < sinks))
    s = (scale * (q @ kx.transpose(2, 3))).masked_fill(~vis, float("-inf"))
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse[..., None])
    o = p @ vx
    dp = d_o @ vx.transpose(2, 3)
    o_sum = o if given_o is None else given_o.double().permute(0, 2, 1, 3)
    ds = scale * p * (dp - (d_o * o_sum).sum(-1, keepdim=True))
    dq, dkx, dvx = ds @ kx, ds.transpose(2, 3) @ q, p.transpose(2, 3) @ d_o
    group = lambda x: x.reshape(B, Hq // rep, rep, T, dk).sum(2)  # noqa: E731
    back = lambda x: x.permute(0, 2, 1, 3)  # noqa: E731
    return back(o), lse, back(dq), back(group(dkx)), back(group(dvx))


def bwd_form(case, dk, dtype):
    """Which launch takes a whole backward of these sizes."""
    B, T, Hq, Hkv, causal, window, sinks = case
    code = _lib.PK_F32 if dtype == torch.float32 else _lib.PK_BF16
    form = _lib.lib().pk_bwd_of_shape(ctypes.byref(_lib.AttnShape(B, T, Hq, Hkv, dk, int(causal), window, sinks, 1.0, code, code)))
    return "SCALAR" if form < 0 else ("APART", "SPLIT", "SPLIT_JOINED", "JOINED", "F32_SPLIT", "F32_PARTS", "F32_PARTS_ALL")[form]


def run_attention(B, T, Hq, Hkv, dk, dtype, causal, window, sinks, grad_dtype=torch.float32):
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    q, d_o = (torch.randn((B, T, Hq, dk), generator=gen, device="cuda").to(dtype) for _ in range(2))
    k, v = (torch.randn((B, T, Hkv, dk), generator=gen, device="cuda").to(dtype) for _ in range(2))
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    got = (o, lse) + ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal, window, sinks, grad_dtype=grad_dtype)
    return got, exact_attention(q, k, v, d_o, scale, causal, window, sinks)


def errors(got, want):
    """Largest difference over the reference's largest value (at least 0.5: a single token has no dQ), per output."""
    return [float((g.double() - w).abs().max()) / max(float(w.abs().max()), 0.5) for g, w in zip(got, want)]


# Workgroups whose wavefronts split the keys or queries: lengths around the 32-row tile, fewer tiles than wavefronts and a
# remainder after dealing them to four and eight, one head and several, units that do not divide by the 8 XCDs.
SPLIT_CASES = [(1, 1, 1, 1, True, 0, 0), (1, 33, 1, 1, True, 0, 0), (3, 159, 1, 1, True, 0, 0), (1, 161, 3, 3, False, 0, 0),
               (1, 300, 5, 5, True, 0, 0), (1, 511, 7, 1, True, 0, 0), (2, 417, 9, 3, True, 0, 0), (1, 700, 2, 2, True, 37, 5),
               (1, 1100, 1, 1, True, 64, 33)]


@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("case", SPLIT_CASES, ids=lambda c: "B%d_T%d_H%d_%d_c%d_w%d_s%d" % c)
def test_split_kernels_of_small_launches(case, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    e = errors(*run_attention(B, T, Hq, Hkv, dk, torch.bfloat16, causal, window, sinks))
    assert max(e) < 1e-2, e


# Head sizes that are no 64 or 128: each multiple of 8 around the padded sizes 32, 64, 96, 128; launches small enough for
# split tiles and large enough for four rows of wavefronts per tile. P and dS keep all their bits there, so fp32 dV is held to
# 2e-5 where the bf16 operand of head_dim 64 / 128 would leave 4e-3; dQ and dK carry the rounding of the bf16 O in
# rowsum(dO .* O).
@pytest.mark.parametrize("dk", [8, 24, 32, 40, 56, 72, 80, 96, 104, 120])
@pytest.mark.parametrize("case", [(1, 200, 3, 1, True, 0, 0), (2, 77, 4, 2, False, 0, 0), (5, 97, 64, 64, True, 0, 0),
                                  (9, 130, 28, 28, True, 40, 3)], ids=lambda c: "B%d_T%d_H%d_%d_c%d_w%d_s%d" % c)
def test_head_sizes_between_the_usual_ones(case, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    e = errors(*run_attention(B, T, Hq, Hkv, dk, torch.bfloat16, causal, window, sinks))
    assert e[0] < 5e-3 and e[1] < 1e-5 and max(e[2:4]) < 5e-3 and e[4] < 2e-5, e


# ... and against the scalar kernels, which take the same values in rows that are not 16-byte aligned and form P and dS in
# fp32: with the O that both are given in the exact rowsum too, what is left is fp32 rounding in one order of summation or
# another, a few 1e-7 of the gradient's norm either way and 2.5e-6 where P or dS lose bits on the way into a product.
@pytest.mark.parametrize("dk", [8, 24, 40, 80, 96, 120])
@pytest.mark.parametrize("case", [(1, 200, 3, 1, True, 0, 0), (5, 97, 64, 64, True, 0, 0), (2, 1024, 4, 4, True, 0, 0),
                                  (9, 130, 28, 28, True, 40, 3)], ids=lambda c: "B%d_T%d_H%d_%d_c%d_w%d_s%d" % c)
def test_gradients_as_exact_as_the_scalar_kernels(case, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    q, k, v, d_o = (torch.randn((B, T, h, dk), generator=gen, device="cuda").bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    want = exact_attention(q, k, v, d_o, scale, causal, window, sinks, o)[2:]
    norms = []
    for view in (lambda x: x, lambda x: torch.nn.functional.pad(x, (0, 1))[..., :dk]):
        got = ops.attn_bwd(*(view(x) for x in (q, k, v, o)), lse, view(d_o), scale, causal, window, sinks, grad_dtype=torch.float32)
        norms.append([float((g.double() - w).norm() / w.norm()) for g, w in zip(got, want)])
    assert all(a < 1.25 * b + 1e-7 for a, b in zip(*norms)), norms


# The same of fp32 tensors: head_dim 32 / 64 / 128 in launches small enough for the split kernels (four and eight
# wavefronts, query heads dealt to several workgroups), and sizes between them at any launch size.
F32_CASES = [(c, dk) for c in SPLIT_CASES for dk in (32, 64, 128)]
F32_CASES += [(c, dk) for c in [(1, 200, 3, 1, True, 0, 0), (2, 77, 4, 2, False, 0, 0), (5, 97, 64, 64, True, 0, 0), (9, 130, 28, 28, True, 40, 3)]
              for dk in (4, 20, 48, 80, 100, 124)]
F32_CASES += [((1, 1100, 8, 2, True, 0, 0), 64), ((1, 1100, 8, 2, True, 300, 4), 32)]


@pytest.mark.parametrize("case,dk", F32_CASES, ids=lambda c: "B%d_T%d_H%d_%d_c%d_w%d_s%d" % c if isinstance(c, tuple) else f"d{c}")
def test_fp32_split_kernels(case, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    e = errors(*run_attention(B, T, Hq, Hkv, dk, torch.float32, causal, window, sinks))
    assert max(e) < 5e-6, e


# fp32 values as three bf16 parts, in launches with the blocks for it: both forms of every kernel, lengths around the 32-row tile
# and the 64- and 128-row blocks, fewer tiles than groups of wavefronts, padded columns, dealt heads and dealt sink tails. What is
# left is fp32 rounding: of a score, of its exponential, and once a tile of the sums, a few times 6e-8 of the norm.
PARTS_CASES = [(20, 161, 11, 11, True, 0, 0), (64, 33, 9, 9, False, 0, 0), (7, 577, 16, 8, True, 0, 0), (13, 511, 16, 16, False, 0, 0),
               (3, 1100, 16, 4, True, 0, 0), (12, 383, 8, 8, True, 37, 5), (1, 2500, 14, 2, True, 0, 0), (10, 1411, 8, 8, True, 33, 9),
               (40, 129, 16, 16, True, 0, 0)]


@pytest.mark.parametrize("dk", [4, 24, 32, 44, 64, 80, 96, 100, 128])
@pytest.mark.parametrize("case", PARTS_CASES, ids=lambda c: "B%d_T%d_H%d_%d_c%d_w%d_s%d" % c)
def test_fp32_as_three_parts(case, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    got, want = run_attention(B, T, Hq, Hkv, dk, torch.float32, causal, window, sinks)
    e = [float((g.double() - w).norm() / w.norm()) for g, w in zip(got, want)]
    assert max(e) < 1e-6, e


def test_fp32_as_three_parts_over_the_range_of_fp32():
    """Columns of V from 1e-25 to 1e35 (P reaches 2^6 and their sum the number of keys), each exact at its own size; a NaN reaches
    what it should."""
    B, T, H, dk = 24, 200, 8, 64
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn((B, T, H, dk), generator=gen, device="cuda") for _ in range(3))
    size = torch.logspace(-25, 35, dk, device="cuda")
    v = v * size
    v[3, 150, 2, 7] = float("nan")
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, _ = ops.attn_fwd(q, k, v, scale)
    p = torch.softmax((scale * (q.double().permute(0, 2, 1, 3) @ k.double().permute(0, 2, 3, 1).contiguous()))
                      .masked_fill(torch.ones(T, T, device="cuda").triu(1).bool(), float("-inf")), -1)
    want = (p @ v.double().nan_to_num(nan=0.0).permute(0, 2, 1, 3).contiguous()).permute(0, 2, 1, 3)
    bad = torch.isnan(o)
    assert bad[3, 150:, 2, 7].all() and int(bad.sum()) == int(bad[3, :, 2, 7].sum())
    good = torch.ones(dk, dtype=torch.bool, device="cuda")
    good[7] = False
    d = (o.double() - want).reshape(-1, dk).norm(dim=0) / want.reshape(-1, dk).norm(dim=0)
    assert float(d[good].max()) < 1e-6, d


def seen(T, key, causal, window, sinks):
    """Which queries see `key`, as a mask over [B, T, H, dk] tensors."""
    i = torch.arange(T, device="cuda")
    vis = (i >= key) if causal else torch.ones_like(i, dtype=torch.bool)
    if window > 0 and key >= sinks:
        vis = vis & (i < key + window)
    return vis.view(1, T, 1, 1)


# launches that take the three-part kernels: both forms, every padded head size, bands, a dealt sink tail, groups of heads, dealt out too
RANGE_CASES = [((24, 200, 8, 8, True, 0, 0), 64), ((5, 4096, 4, 4, True, 0, 0), 64), ((13, 511, 16, 8, False, 0, 0), 96), ((12, 383, 8, 8, True, 37, 5), 32),
               ((20, 161, 11, 11, True, 0, 0), 128), ((7, 577, 16, 8, True, 0, 0), 44), ((10, 1411, 8, 8, True, 33, 9), 64), ((1, 2500, 14, 2, True, 0, 0), 64),
               ((3, 1100, 16, 4, True, 0, 0), 100)]
# ... and the joined launch of the backward above 64 columns
RANGE_CASES += [((3, 577, 8, 8, False, 0, 0), 96), ((4, 640, 8, 8, True, 0, 0), 96), ((6, 321, 9, 9, True, 33, 17), 96),
                ((3, 577, 8, 8, False, 0, 0), 128), ((2, 577, 19, 19, True, 0, 0), 128), ((6, 321, 9, 9, True, 33, 17), 128)]


def test_range_cases_reach_every_form_of_the_backward():
    forms = {(bwd_form(case, dk, torch.float32), max(32, (dk + 31) // 32 * 32), case[4]) for case, dk in RANGE_CASES}
    assert {f[:2] for f in forms} >= {("APART", d) for d in (64, 96, 128)} | {("F32_PARTS", d) for d in (64, 96, 128)} | {("F32_PARTS_ALL", d) for d in (32, 96, 128)}
    assert {("F32_PARTS", 96, False), ("F32_PARTS", 128, False)} <= forms


@pytest.mark.parametrize("case,dk", RANGE_CASES, ids=str)
def test_three_parts_keep_infinities(case, dk):
    """The reference's arithmetic over the visible keys (src/ops.cpp:879-932). A key whose scores are all -inf has no weight, and only dQ
    shows it, in the column where it is infinite: 0 times inf. An infinite value makes its column of O infinite in the rows that see it
    and in no others. Finite results to the bound of the test above."""
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    q, k, v, d_o = (torch.randn((B, T, h, dk), generator=gen, device="cuda") for h in (Hq, Hkv, Hkv, Hq))
    q[..., 1] = -q[..., 1].abs() - 0.1
    key, scale = 1 if sinks > 1 else T // 3, float(np.float32(1.0 / np.sqrt(dk)))
    sees = seen(T, key, causal, window, sinks)
    k_inf, k_zero = k.clone(), k.clone()
    k_inf[:, key, :, 1], k_zero[:, key] = float("inf"), 0.0
    o, lse = ops.attn_fwd(q, k_inf, v, scale, causal, window, sinks)
    got = [o, lse, *ops.attn_bwd(q, k_inf, v, o, lse, d_o, scale, causal, window, sinks)]
    want = list(exact_attention(q, k_inf, v, d_o, scale, causal, window, sinks))
    want[2] = torch.where(sees, want[2], exact_attention(q, k_zero, v, d_o, scale, causal, window, sinks)[2])
    assert torch.equal(torch.isnan(got[2][..., 1]), sees[..., 0].expand(B, T, Hq))
    got[2], want[2] = (torch.where(sees & (torch.arange(dk, device="cuda") == 1), 0.0, x) for x in (got[2], want[2]))
    e = [float((g.double() - w).norm() / w.norm()) for g, w in zip(got, want)]
    assert max(e) < 1e-6, e

    v_inf, v_zero = v.clone(), v.clone()
    v_inf[:, key, :, 3], v_zero[:, key, :, 3] = float("inf"), 0.0
    o, lse = ops.attn_fwd(q, k, v_inf, scale, causal, window, sinks)
    want = exact_attention(q, k, v_zero, d_o, scale, causal, window, sinks)
    there = sees & (torch.arange(dk, device="cuda") == 3)
    assert bool((o == float("inf")).eq(there).all())
    e = [float((g.double() - w).norm() / w.norm()) for g, w in zip((torch.where(there, 0.0, o), lse), (torch.where(there, 0.0, want[0]), want[1]))]
    assert max(e) < 1e-6, e


@pytest.mark.parametrize("case,dk", RANGE_CASES, ids=str)
def test_three_parts_hold_what_the_weights_keep_in_range(case, dk):
    """Values up to the largest of fp32: O is a weighted mean of them, whatever their sum under weights of up to 2^6 would be, and
    values past the largest bf16 have no rounded first part. Bound as above."""
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    q, k, d_o = (torch.randn((B, T, h, dk), generator=gen, device="cuda") for h in (Hq, Hkv, Hq))
    v = torch.rand((B, T, Hkv, dk), generator=gen, device="cuda") * 3.4e38
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, _ = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    want = exact_attention(q, k, v * 2.0 ** -40, d_o, scale, causal, window, sinks)[0]
    e = float((o.double() * 2.0 ** -40 - want).norm() / want.norm())
    assert e < 1e-6, e


def test_three_parts_round_single_products_as_fp32_does():
    """Scores of one product each, and rows that see one key (a window of one): LSE is that product. A product of three parts leaves out
    2^-8 x 2^-17 of it twice and 2^-34; the sum of the others is off by a unit of its last place at most, 2^-23. The factors are near
    the powers of two, where what is left out weighs most (general ones on the fp32 instruction: 1.3e-7)."""
    B, T, H, dk = 4, 1024, 8, 64
    gen = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.zeros((B, T, H, dk), device="cuda") for _ in range(3))
    q[..., 5] = (1 + 0.1 * torch.rand((B, T, H), generator=gen, device="cuda")) * 1024
    k[..., 5] = -(1 + 0.1 * torch.rand((B, T, H), generator=gen, device="cuda")) * 1024
    _, lse = ops.attn_fwd(q, k, v, 1.0, True, 1, 0)
    want = (q[..., 5].double() * k[..., 5].double()).permute(0, 2, 1)
    e = float(((lse.double() - want) / want).abs().max())
    assert e <= (3 + 2.0 ** -9) * 2.0 ** -24, e


@pytest.mark.parametrize("tiny", ["v", "d_o", "k"])
@pytest.mark.parametrize("case,dk", RANGE_CASES, ids=str)
def test_three_parts_of_tiny_tensors(case, dk, tiny):
    """Values below 1e-33, whose last parts are below the range of bf16: results as exact as of others. Bound as above."""
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    x = {n: torch.randn((B, T, h, dk), generator=gen, device="cuda") for n, h in (("q", Hq), ("k", Hkv), ("v", Hkv), ("d_o", Hq))}
    x[tiny] *= 2.0 ** -120
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(x["q"], x["k"], x["v"], scale, causal, window, sinks)
    got = (o, lse, *ops.attn_bwd(x["q"], x["k"], x["v"], o, lse, x["d_o"], scale, causal, window, sinks))
    e = [float((g.double() - w).norm() / w.norm()) for g, w in zip(got, exact_attention(x["q"], x["k"], x["v"], x["d_o"], scale, causal, window, sinks))]
    assert max(e) < 1e-6, e


# Launches of the whole backward in three parts where dQ or dK/dV by itself would be on the fp32 instruction: every padded head size, masked
# and not, bands, groups of heads, dealt out too
WHOLE_RANGE_CASES = [((12, 383, 8, 8, True, 37, 5), 32), ((5, 577, 8, 8, False, 0, 0), 20), ((4, 313, 16, 16, True, 0, 0), 64), ((7, 65, 16, 8, True, 0, 0), 44),
                     ((6, 321, 9, 9, True, 33, 17), 80), ((1, 710, 8, 8, False, 0, 0), 96), ((2, 641, 13, 13, True, 0, 0), 128),
                     ((1, 2113, 8, 2, True, 0, 0), 100), ((1, 710, 8, 8, False, 0, 0), 128)]


@pytest.mark.parametrize("tensors", ["kq", "q", "k", "v", "d_o"])
@pytest.mark.parametrize("case,dk", WHOLE_RANGE_CASES, ids=str)
def test_joined_parts_hold_columns_of_every_size(case, dk, tensors):
    """Columns from 2^-120 to 2^20 of one tensor, or one of K at 2^-120 whose scores one of Q at 2^120 makes ordinary: every column of every
    gradient exact at its own size, from the O and LSE of float64. Bound as of test_fp32_as_three_parts."""
    assert bwd_form(case, dk, torch.float32) == "F32_PARTS_ALL"
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    x = {n: torch.randn((B, T, h, dk), generator=gen, device="cuda") for n, h in (("q", Hq), ("k", Hkv), ("v", Hkv), ("d_o", Hq))}
    if tensors == "kq":
        x["q"][..., 2] *= 2.0 ** 120
        x["k"][..., 2] *= 2.0 ** -120
    else:
        x[tensors] *= 2.0 ** torch.linspace(-120, 20 if tensors in ("v", "d_o") else 0, dk, device="cuda").round()
        x["d_o"] *= 1.0 if tensors in ("v", "d_o") else 2.0 ** 20  # dQ and dK at 2^-120 of it are in fp32's range
    args = (x["q"], x["k"], x["v"], x["d_o"], float(np.float32(1.0 / np.sqrt(dk))), causal, window, sinks)
    o, lse = (t.float().contiguous() for t in exact_attention(*args)[:2])
    got = ops.attn_bwd(*args[:3], o, lse, *args[3:])
    columns = lambda t: t.double().reshape(-1, dk).norm(dim=0)  # noqa: E731
    e = [float((columns(g.double() - w) / columns(w)).max()) for g, w in zip(got, exact_attention(*args, o)[2:])]
    assert max(e) < 1e-6, e


# dQ and dK/dV in one launch against the two launches of the same call's stages: the forms, and so the order of the sums, may differ,
# nothing else does. Few tiles and remainders, groups of heads dealt out and not, sink tails, the largest launches that go together.
@pytest.mark.parametrize("dtype,dk", [(torch.bfloat16, 24), (torch.bfloat16, 64), (torch.bfloat16, 96), (torch.bfloat16, 128), (torch.float32, 20),
                                      (torch.float32, 64), (torch.float32, 96), (torch.float32, 128)], ids=str)
@pytest.mark.parametrize("case", [(1, 1, 1, 1, True, 0, 0), (3, 33, 2, 1, False, 0, 0), (2, 129, 7, 1, True, 0, 0), (1, 770, 2, 2, True, 64, 1),
                                  (1, 1300, 7, 1, True, 100, 32), (5, 200, 4, 4, True, 0, 0), (1, 97, 64, 8, True, 0, 0)], ids=str)
def test_backward_in_one_launch(case, dtype, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    q, k, v, d_o = (torch.randn((B, T, h, dk), generator=gen, device="cuda").to(dtype) for h in (Hq, Hkv, Hkv, Hq))
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    one = ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal, window, sinks, grad_dtype=torch.float32)
    bufs = [torch.empty(x.shape, dtype=torch.float32, device="cuda") for x in (q, k, v)]
    ws = torch.empty(ops.bwd_workspace_bytes(q, k, torch.float32, window, sinks), dtype=torch.uint8, device="cuda")
    for stages in (ops.BWD_DELTA | ops.BWD_DQ, ops.BWD_DKDV):
        ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal, window, sinks, grad_dtype=torch.float32, out=(*bufs, ws), stages=stages)
    # bf16 operands of P and dS at 64 and 128 columns: 2^-9 of a term each, of 4 standard deviations at most
    tol = 1e-2 if dtype == torch.bfloat16 and dk in (64, 128) else 5e-6
    for a, b in zip(one, bufs):
        assert float((a - b).abs().max()) <= tol * max(float(b.abs().max()), 0.5)
    e = errors((o, lse) + tuple(one), exact_attention(q, k, v, d_o, scale, causal, window, sinks))
    assert max(e) < (1e-2 if dtype == torch.bfloat16 else 5e-6), e


# fp32 blocks of 64 keys and of 64 queries in one launch behind one of delta: one row past a block and a tile, more ranks than heads, groups
# whose heads are dealt out, units that do not divide by the 8 XCDs, the shortest chains and the most blocks that go together.
@pytest.mark.parametrize("dk", [4, 32, 44, 64, 80, 96, 100, 128])
@pytest.mark.parametrize("case", [(18, 33, 16, 16, True, 0, 0), (7, 65, 16, 8, True, 0, 0), (9, 129, 14, 2, True, 0, 0), (2, 641, 13, 13, True, 0, 0),
                                  (5, 577, 8, 8, False, 0, 0), (1, 2113, 8, 2, True, 0, 0), (40, 257, 3, 3, True, 0, 0), (6, 321, 9, 9, True, 33, 17),
                                  (1, 1100, 11, 11, True, 100, 0), (8, 471, 6, 6, True, 91, 4), (7, 129, 14, 2, True, 0, 0), (3, 577, 8, 8, False, 0, 0),
                                  (20, 257, 3, 3, True, 0, 0)], ids=str)
def test_fp32_backward_of_joined_blocks(case, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    past = dk > 64 and case[:2] in ((9, 129), (5, 577), (40, 257))  # the sizes past the last one that goes together
    assert bwd_form(case, dk, torch.float32).startswith("APART" if past else "F32_PARTS")
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    cut = lambda x: (x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:])  # noqa: E731
    q, k, v = cut(torch.randn((B, T, Hq + 2 * Hkv, dk), generator=gen, device="cuda"))
    d_o = torch.randn((B, Hq, T, dk), generator=gen, device="cuda").permute(0, 2, 1, 3)
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    one = ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal, window, sinks)
    again = ops.attn_bwd(*(x.contiguous() for x in (q, k, v)), o, lse, d_o.contiguous(), scale, causal, window, sinks)
    assert all(torch.equal(x, y) for x, y in zip(one, again))
    want = exact_attention(q, k, v, d_o, scale, causal, window, sinks)[2:]
    e = [float((g.double() - w).norm() / w.norm()) for g, w in zip(one, want)]
    assert max(e) < 1e-6, e  # as test_fp32_as_three_parts


# bf16 blocks of 128 keys and of 128 queries in one launch: one tile and one row past it, one row past a block, rows past the end in the last
# tile that delta is formed of, groups whose heads are dealt out, units that do not divide by the 8 XCDs; O a view as the others are.
@pytest.mark.parametrize("dk", [8, 32, 40, 64, 80, 96])
@pytest.mark.parametrize("case", [(17, 33, 16, 16, True, 0, 0), (9, 65, 16, 8, True, 0, 0), (13, 129, 8, 8, False, 0, 0), (11, 193, 14, 2, True, 0, 0),
                                  (5, 577, 9, 3, True, 0, 0), (2, 1025, 16, 4, True, 0, 0), (3, 700, 9, 9, False, 0, 0), (9, 321, 9, 9, True, 33, 17),
                                  (2, 1100, 12, 12, True, 100, 0), (1, 1025, 36, 9, True, 0, 0), (4, 700, 9, 9, False, 0, 0)], ids=str)
def test_bf16_backward_of_joined_blocks(case, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    below = (dk < 64 and case[:2] == (2, 1025)) or (dk > 64 and case[:2] == (3, 700))  # sizes below the first one that goes together
    assert bwd_form(case, dk, torch.bfloat16) == ("APART" if below else "SPLIT_JOINED")
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    cut = lambda x: (x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:])  # noqa: E731
    q, k, v = cut(torch.randn((B, T, Hq + 2 * Hkv, dk), generator=gen, device="cuda").bfloat16())
    d_o = torch.randn((B, Hq, T, dk), generator=gen, device="cuda").bfloat16().permute(0, 2, 1, 3)
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    o_view = torch.full((B, T, 2 * Hq, dk), float("nan"), device="cuda").bfloat16()[:, :, :Hq]
    o_view.copy_(o)
    one = ops.attn_bwd(q, k, v, o_view, lse, d_o, scale, causal, window, sinks, grad_dtype=torch.float32)
    again = ops.attn_bwd(*(x.contiguous() for x in (q, k, v, o)), lse, d_o.contiguous(), scale, causal, window, sinks, grad_dtype=torch.float32)
    assert all(torch.equal(x, y) for x, y in zip(one, again))
    want = exact_attention(q, k, v, d_o, scale, causal, window, sinks, o)[2:]
    e = [float((g.double() - w).norm() / w.norm()) for g, w in zip(one, want)]
    # 64 columns: P and dS as one bf16 operand, 2^-9 of a term; the others keep all their bits
    assert max(e) < (4e-3 if dk == 64 else 2e-6), e


@pytest.mark.parametrize("case", [(4, 150, 16, 16, True, 0, 0), (2, 1104, 16, 8, True, 0, 0), (14, 423, 2, 2, False, 0, 0), (9, 65, 16, 8, True, 0, 0),
                                  (31, 64, 4, 4, True, 0, 0), (40, 200, 2, 2, True, 0, 0)], ids=str)
def test_joined_blocks_round_dp_as_the_launches_do(case):
    """V the same in every row: dS is zero, and dQ and dK are what the sums of dP and delta are rounded by. The launches by themselves subtract delta
    from the finished sum, and the joined one rounds no more than they do (a sum that starts from -delta is off by two to four times as much). Its dK/dV
    forms delta in another order, so the same roundings come out up to 1.3 times as large there."""
    B, T, Hq, Hkv, causal, window, sinks = case
    dk, gen = 64, torch.Generator(device="cuda").manual_seed(T)
    q, k, d_o = (torch.randn((B, T, h, dk), generator=gen, device="cuda").bfloat16() for h in (Hq, Hkv, Hq))
    v = torch.full((B, T, Hkv, dk), 4096.0, device="cuda").bfloat16()
    o, lse = ops.attn_fwd(q, k, v, 0.125, causal, window, sinks)
    assert bwd_form(case, dk, torch.bfloat16) == "SPLIT_JOINED" and bool((o == 4096).all())
    one = ops.attn_bwd(q, k, v, o, lse, d_o, 0.125, causal, window, sinks, grad_dtype=torch.float32)
    bufs = [torch.empty(x.shape, dtype=torch.float32, device="cuda") for x in (q, k, v)]
    ws = torch.empty(ops.bwd_workspace_bytes(q, k, torch.float32, window, sinks), dtype=torch.uint8, device="cuda")
    ops.attn_bwd(q, k, v, o, lse, d_o, 0.125, causal, window, sinks, grad_dtype=torch.float32, out=(*bufs, ws), stages=ops.BWD_DELTA | ops.BWD_DQ)
    assert float(one[0].norm()) <= 1.01 * float(bufs[0].norm())
    ops.attn_bwd(q, k, v, o, lse, d_o, 0.125, causal, window, sinks, grad_dtype=torch.float32, out=(*bufs, ws), stages=ops.BWD_DKDV)
    assert float(one[1].norm()) <= 1.6 * float(bufs[1].norm())


# The same at head_dim 128, blocks of 64 keys and of 128 queries: one row past a tile and past either block, an odd number of blocks of keys,
# bands with and without sinks, both gradient types.
@pytest.mark.parametrize("grad", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("case", [(9, 33, 9, 9, True, 0, 0), (11, 65, 5, 5, False, 0, 0), (13, 129, 9, 9, True, 0, 0), (4, 577, 7, 7, True, 0, 0), (3, 700, 6, 6, False, 0, 0),
                                  (1, 1793, 12, 12, True, 0, 0), (6, 321, 9, 9, True, 33, 17), (1, 4200, 3, 3, True, 100, 0), (3, 161, 28, 4, True, 0, 0),
                                  (1, 700, 14, 2, False, 0, 0), (2, 450, 16, 4, True, 60, 0), (1, 450, 16, 4, True, 60, 0), (2, 450, 8, 4, True, 60, 0)], ids=str)
def test_bf16_backward_of_joined_blocks_at_128(case, grad):
    B, T, Hq, Hkv, causal, window, sinks = case
    assert bwd_form(case, 128, torch.bfloat16) == ("APART" if case[:3] == (2, 450, 16) else "JOINED")  # (its group of four is not dealt out)
    gen = torch.Generator(device="cuda").manual_seed(T)
    cut = lambda x: (x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:])  # noqa: E731
    q, k, v = cut(torch.randn((B, T, Hq + 2 * Hkv, 128), generator=gen, device="cuda").bfloat16())
    d_o = torch.randn((B, Hq, T, 128), generator=gen, device="cuda").bfloat16().permute(0, 2, 1, 3)
    scale = float(np.float32(1.0 / np.sqrt(128)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    o_view = torch.full((B, T, 2 * Hq, 128), float("nan"), device="cuda").bfloat16()[:, :, :Hq]
    o_view.copy_(o)
    one = ops.attn_bwd(q, k, v, o_view, lse, d_o, scale, causal, window, sinks, grad_dtype=grad)
    again = ops.attn_bwd(*(x.contiguous() for x in (q, k, v, o)), lse, d_o.contiguous(), scale, causal, window, sinks, grad_dtype=grad)
    assert all(torch.equal(x, y) for x, y in zip(one, again))
    want = exact_attention(q, k, v, d_o, scale, causal, window, sinks, o)[2:]
    e = [float((g.double() - w).norm() / w.norm()) for g, w in zip(one, want)]
    assert max(e) < 4e-3, e  # P and dS as one bf16 operand, and the gradient's own rounding


# A training loop that keeps no tensors it can do without: dQ where O was, dK and dV where K and V were. Small launches and large ones,
# groups of heads dealt out, dealt sink tails, head sizes of every kernel family. The same bits as dQ and then dK/dV into buffers of
# their own, which read what they read in this order.
@pytest.mark.parametrize("dtype,dk", [(torch.bfloat16, 24), (torch.bfloat16, 64), (torch.bfloat16, 128), (torch.float32, 20), (torch.float32, 64),
                                      (torch.float32, 128)], ids=str)
@pytest.mark.parametrize("case", [(1, 97, 4, 4, True, 0, 0), (2, 129, 7, 1, True, 0, 0), (1, 770, 2, 2, True, 64, 1), (3, 200, 4, 4, False, 0, 0),
                                  (4, 1024, 8, 8, True, 0, 0), (16, 512, 8, 4, True, 0, 0), (8, 700, 16, 16, True, 100, 4)], ids=str)
def test_gradients_in_the_place_of_inputs(case, dtype, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    q, k, v, d_o = (torch.randn((B, T, h, dk), generator=gen, device="cuda").to(dtype) for h in (Hq, Hkv, Hkv, Hq))
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    want = [torch.empty_like(x) for x in (q, k, v)]
    ws = torch.empty(ops.bwd_workspace_bytes(q, k, window=window, sinks=sinks), dtype=torch.uint8, device="cuda")
    for stages in (ops.BWD_DELTA | ops.BWD_DQ, ops.BWD_DKDV):
        ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal, window, sinks, out=(*want, ws), stages=stages)
    got = ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal, window, sinks, out=(o, k, v, ws))
    assert all(a.data_ptr() == b.data_ptr() for a, b in zip(got, (o, k, v)))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


# As a model calls them: q, k and v are slices of one projection, of every other sequence of a longer batch, dO is a transposed view and
# the gradients go into slices of one buffer. The same kernels as of contiguous tensors, so the same bits: three parts, one launch for
# the backward, wavefronts that own their rows at head_dim 64.
@pytest.mark.parametrize("case,dtype,dk", [((24, 200, 8, 8, True, 0, 0), torch.float32, 64), ((13, 511, 16, 8, False, 0, 0), torch.float32, 96),
                                           ((12, 383, 8, 8, True, 37, 5), torch.float32, 32), ((20, 161, 11, 11, True, 0, 0), torch.float32, 128),
                                           ((3, 1100, 16, 4, True, 0, 0), torch.float32, 44)] +
                         [((2, 129, 7, 1, True, 0, 0), t, d) for t, d in [(torch.bfloat16, 24), (torch.bfloat16, 64), (torch.bfloat16, 128), (torch.float32, 20),
                                                                          (torch.float32, 64), (torch.float32, 128)]] +
                         [((1, 770, 2, 2, True, 64, 1), t, 64) for t in (torch.bfloat16, torch.float32)] +
                         [(c, torch.bfloat16, 64) for c in [(16, 512, 8, 8, True, 0, 0), (6, 777, 12, 12, False, 0, 0), (3, 1889, 16, 16, True, 69, 16),
                                                            (2, 2049, 14, 2, True, 0, 0), (8, 700, 16, 8, True, 128, 0)]], ids=str)
def test_strided_tensors_give_the_bits_of_contiguous_ones(case, dtype, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    cut = lambda x: (x[:, :, :Hq], x[:, :, Hq:Hq + Hkv], x[:, :, Hq + Hkv:])  # noqa: E731
    q, k, v = cut(torch.randn((2 * B, T, Hq + 2 * Hkv, dk), generator=gen, device="cuda").to(dtype)[::2])
    d_o = torch.randn((B, Hq, T, dk), generator=gen, device="cuda").to(dtype).permute(0, 2, 1, 3)
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    ws = torch.empty(ops.bwd_workspace_bytes(q, k, window=window, sinks=sinks), dtype=torch.uint8, device="cuda")
    results = []
    for view in (lambda x: x, lambda x: x.contiguous()):
        a = [view(x) for x in (q, k, v)]
        o, lse = ops.attn_fwd(*a, scale, causal, window, sinks)
        out = [view(x) for x in cut(torch.full((B, T, Hq + 2 * Hkv, dk), float("nan"), device="cuda").to(dtype))]
        results.append((o, lse, *ops.attn_bwd(*a, o, lse, view(d_o), scale, causal, window, sinks, out=(*out, ws))))
    assert not q.is_contiguous() and not d_o.is_contiguous()
    assert all(torch.equal(x, y) for x, y in zip(*results))
    e = errors(results[0], exact_attention(q, k, v, d_o, scale, causal, window, sinks))
    assert max(e) < (1e-2 if dtype == torch.bfloat16 else 5e-6), e


# bf16 at head_dim 64 in launches that fill the chip: rows owned by wavefronts, two or four to a workgroup, tiles of 32 and 64; lengths
# around the tiles and blocks, the shortest that come here, bands with and without sinks (dealt out and left whole), dealt heads, no mask.
@pytest.mark.parametrize("case", [(16, 512, 8, 8, True, 0, 0), (64, 65, 8, 8, True, 0, 0), (20, 399, 8, 8, True, 0, 0), (2, 2049, 14, 2, True, 0, 0),
                                  (6, 777, 12, 12, False, 0, 0), (40, 129, 8, 4, False, 0, 0), (3, 1889, 16, 16, True, 69, 16),
                                  (2, 2500, 16, 16, True, 200, 0), (8, 700, 16, 8, True, 128, 0), (4, 300, 16, 16, True, 33, 3),
                                  (1, 1100, 32, 32, True, 0, 0)], ids=str)
def test_rows_owned_by_wavefronts_at_head_dim_64(case):
    e = errors(*run_attention(*case[:4], 64, torch.bfloat16, *case[4:]))
    assert max(e) < 1e-2, e


# Either side of the lines between the two geometries of the 32-key dK/dV kernel: one round of the chip and one head more, two
# nearly whole rounds, and with a band and sink keys whose queries are dealt out or left whole.
@pytest.mark.parametrize("case,dk", [((32, 200, 8, 8, True, 0, 0), 64), ((33, 200, 4, 4, True, 0, 0), 64), ((16, 200, 8, 8, True, 0, 0), 64),
                                     ((17, 200, 8, 8, True, 0, 0), 64), ((16, 512, 8, 8, True, 0, 0), 64), ((20, 320, 8, 8, False, 0, 0), 64),
                                     ((32, 160, 8, 8, False, 0, 0), 64), ((32, 96, 8, 8, True, 0, 0), 128), ((16, 256, 8, 8, True, 0, 0), 128),
                                     ((8, 300, 8, 8, True, 100, 0), 64), ((10, 1000, 8, 8, True, 64, 4), 64), ((8, 1000, 8, 8, True, 32, 4), 64),
                                     ((5, 1000, 8, 8, True, 300, 0), 64)], ids=str)
def test_lines_between_the_dkdv_geometries(case, dk):
    e = errors(*run_attention(*case[:4], dk, torch.bfloat16, *case[4:]))
    assert max(e) < 1e-2, e


# Either side of the lines between the split kernels and the others at the usual head sizes: the shortest sequences, one and
# two rounds of blocks, and groups of heads.
@pytest.mark.parametrize("case,dtype,dk", [(c, torch.bfloat16, d) for c in [(1, 90, 8, 8, True, 0, 0), (2, 177, 9, 9, True, 0, 0), (3, 322, 16, 16, True, 0, 0),
                                           (2, 350, 13, 13, True, 0, 0), (1, 1700, 10, 10, False, 0, 0), (2, 40, 4, 2, True, 13, 0), (2, 60, 14, 2, True, 20, 2)]
                                           for d in (64, 128)] +
                                          [(c, torch.float32, d) for c in [(2, 26, 6, 6, True, 0, 0), (9, 30, 8, 2, False, 0, 0), (24, 32, 6, 3, True, 0, 0),
                                           (30, 96, 4, 4, True, 0, 0)] for d in (32, 64, 128)] + [((50, 200, 8, 4, True, 0, 0), torch.float32, 64)], ids=str)
def test_lines_between_split_and_unsplit_launches(case, dtype, dk):
    e = errors(*run_attention(*case[:4], dk, dtype, *case[4:]))
    assert max(e) < (1e-2 if dtype == torch.bfloat16 else 5e-6), e


# Query heads that share KV heads where the launch is one of a kernel that walks the group in one workgroup: the workspace is
# the row sums alone, and the entry point with the library's own scratch runs the same kernels.
@pytest.mark.parametrize("case,dtype,dk", [((31, 256, 16, 4, True, 0, 0), torch.bfloat16, 64), ((67, 64, 8, 2, False, 0, 0), torch.bfloat16, 128),
                                           ((4, 1100, 16, 4, True, 0, 0), torch.float32, 128)], ids=str)
def test_query_groups_without_partial_sums(case, dtype, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    q, k, v, d_o = (torch.randn((B, T, h, dk), generator=torch.Generator(device="cuda").manual_seed(i), device="cuda").to(dtype)
                    for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    assert ops.bwd_workspace_bytes(q, k) == 4 * B * Hq * T
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal)
    got = ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal)
    assert all(torch.equal(a, b) for a, b in zip(got, ops.attn_bwd_static(q, k, v, o, lse, d_o, scale, causal)))
    e = errors((o, lse) + got, exact_attention(q, k, v, d_o, scale, causal, window, sinks))
    assert max(e) < (1e-2 if dtype == torch.bfloat16 else 5e-6), e


# The queries past the sink keys' band dealt to workgroups of their own: one chunk and a short last one, all 32 sink rows,
# query heads dealt as well, blocks of 32 keys and (bf16, head_dim 48, many of them) of 128.
@pytest.mark.parametrize("dtype,dk", [(torch.bfloat16, 48), (torch.bfloat16, 64), (torch.bfloat16, 128), (torch.float32, 32),
                                      (torch.float32, 64), (torch.float32, 128)], ids=str)
@pytest.mark.parametrize("case", [(1, 770, 2, 2, True, 64, 1), (1, 1300, 7, 1, True, 100, 32), (2, 1411, 4, 2, True, 33, 5),
                                  (9, 1200, 4, 4, True, 40, 16)], ids=lambda c: "B%d_T%d_H%d_%d_c%d_w%d_s%d" % c)
def test_sink_tail_of_the_split_kernels(case, dtype, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    e = errors(*run_attention(B, T, Hq, Hkv, dk, dtype, causal, window, sinks))
    assert max(e) < (1e-2 if dtype == torch.bfloat16 else 5e-6), e


@pytest.mark.parametrize("dtype,dk", [(torch.bfloat16, 64), (torch.bfloat16, 128), (torch.float32, 64), (torch.float32, 48)], ids=str)
@pytest.mark.parametrize("case", [(1, 615, 7, 1, 25, 16), (1, 636, 28, 4, 21, 16), (1, 1300, 14, 2, 114, 1), (3, 300, 7, 1, 20, 4)],
                         ids=lambda c: "B%d_T%d_H%d_%d_w%d_s%d" % c)
def test_sink_keys_of_groups_dealt_out(case, dtype, dk):
    """Query heads of a group dealt to several workgroups under a band with sinks: whether the sink keys' block walks its heads' tail
    itself or pieces of it go to others. Bounds as in the test above."""
    B, T, Hq, Hkv, window, sinks = case
    e = errors(*run_attention(B, T, Hq, Hkv, dk, dtype, True, window, sinks))
    assert max(e) < (1e-2 if dtype == torch.bfloat16 else 5e-6), e


@pytest.mark.parametrize("B,T,Hq,Hkv,dk,window,sinks", [(1, 3050, 7, 1, 64, 1700, 32), (3, 1122, 7, 1, 64, 108, 4), (2, 540, 28, 4, 128, 27, 1),
                                                        (5, 913, 7, 1, 80, 343, 1), (1, 600, 32, 8, 32, 70, 16), (12, 1055, 4, 1, 128, 33, 4)])
def test_fp32_groups_dealt_out_for_their_sink_keys(B, T, Hq, Hkv, dk, window, sinks):
    """Launches that fill the chip undealt, from 96 to 400 blocks of 32 keys. Bound as in the test above."""
    e = errors(*run_attention(B, T, Hq, Hkv, dk, torch.float32, True, window, sinks))
    assert max(e) < 5e-6, e


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (33, 65, 31), (64, 32, 33), (31, 97, 344), (1, 40, 1001), (900, 1030, 70)])
def test_fp32_products(M, N, K, tA, tB):
    """The hand-written fp32 GEMM at the edges of its tiles (32 and, from 640 of those on, 64), of its contraction chunks
    and of the split of the contraction among wavefronts, with and without the sum onto C. Against float64."""
    import ctypes as C

    from paperkiln_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, b = (torch.randn(s, generator=gen, device="cuda") for s in ((K, M) if tA else (M, K), (N, K) if tB else (K, N)))
    c0 = torch.randn((M, N), generator=gen, device="cuda")
    want = (a.double().T if tA else a.double()) @ (b.double().T if tB else b.double())
    for accumulate in (0, 1):
        c = c0.clone()
        _lib.check(_lib.lib().pk_op_gemm(C.c_void_p(a.data_ptr()), tA, C.c_void_p(b.data_ptr()), tB, C.c_void_p(c.data_ptr()),
                                         M, N, K, _lib.PK_F32, _lib.PK_F32, accumulate, None))
        torch.cuda.synchronize()
        err = (c.double() - want - accumulate * c0.double()).abs().max()
        assert err < 4e-7 * (K + 16) ** 0.5 * 4, (accumulate, float(err))


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", [(256, 255, 31), (257, 250, 129), (511, 241, 300), (513, 225, 255), (529, 240, 257), (500, 530, 256), (495, 545, 261)])
def test_fp32_products_of_each_tile(M, N, K, tA, tB):
    """The same around the numbers of 32 x 32 tiles (64, 128, 256) and the lengths (256) at which its tile changes: 16 x 16,
    16 x 32 and 32 x 32 with four and eight wavefronts. The bound: a sum of K products of standard normal numbers, each partial
    sum rounded with a standard deviation of 2.4e-8 of its size sqrt(k), is off by 1.7e-8 K; five times that is below it
    up to K = 350."""
    test_fp32_products(M, N, K, tA, tB)


@pytest.mark.parametrize("M,N,K", [(700, 580, 257), (900, 1030, 300), (513, 640, 1001)])
def test_fp32_weight_gradients_of_wide_tiles(M, N, K):
    """Weight gradients in tiles of 32 x 64, with four and eight wavefronts. The bound: a wavefront's chain is at most 126 sums, each
    rounded with a standard deviation of 0.58 of 2^-24 of a partial sum, which is about a tenth of the sum of the terms' magnitudes
    and seldom a third; five times sqrt(126) 0.58 / 3 of that is below 11."""
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, b, c0 = (torch.randn(s, generator=gen, device="cuda") for s in ((K, M), (K, N), (M, N)))
    for out in (None, c0.clone()):
        got = blockops.matmul(a, b, trans_a=True, out=out)
        base = 0 if out is None else c0.double()
        room = 11 * 2.0 ** -24 * (a.abs().double().T @ b.abs().double() + (0 if out is None else c0.abs().double()))
        assert ((got.double() - (a.double().T @ b.double() + base)).abs() <= room).all()


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("M,N", [(256, 256), (512, 256)])  # up to 64 tiles of 32 x 32, up to 128
def test_long_fp32_products_are_split_eight_ways(M, N, tA, tB):
    """A chain loses terms below half a unit of its sum's last place: with 1 as the first term and 0.9 x 2^-27 ever after (four of them
    in an instruction) the chain that holds the 1 loses all of its others, the K / 8 of one chain of eight, and the chains' sums and
    the rows past a chunk's end are rounded once each."""
    K = 2048
    a, b = (torch.ones(s, device="cuda") for s in ((K, M) if tA else (M, K), (N, K) if tB else (K, N)))
    (a if tA else a.T)[1:] = 0.9 * 2.0 ** -27
    c = blockops.matmul(a, b, bool(tA), bool(tB))
    want = 1 + (K - 1) * 0.9 * 2.0 ** -27
    assert float((c.double() - want).abs().max()) <= (K // 8 + 32) * 0.9 * 2.0 ** -27 + 8 * 2.0 ** -24


@pytest.mark.parametrize("c_dtype", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", [(2, 2, 32), (34, 66, 34), (64, 32, 64), (62, 30, 344), (2, 40, 1002), (126, 130, 700), (1000, 64, 66)])
def test_small_bf16_products(M, N, K, tA, tB, c_dtype):
    """The bf16 GEMM of few tiles at the edges of those (32), of its contraction chunks (an odd length where both operands
    have it as rows) and of the split among four and eight wavefronts, with and without the sum onto C."""
    K += tA
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, b = (torch.randn(s, generator=gen, device="cuda").bfloat16() for s in ((K, M) if tA else (M, K), (N, K) if tB else (K, N)))
    c0 = torch.randn((M, N), generator=gen, device="cuda").to(c_dtype)
    want = (a.double().T if tA else a.double()) @ (b.double().T if tB else b.double())
    for out in (None, c0.clone()):
        got = blockops.matmul(a, b, bool(tA), bool(tB), out_dtype=c_dtype, out=out)
        torch.cuda.synchronize()
        exact = want + (0 if out is None else c0.double())
        err = ((got.double() - exact).abs() - (exact.abs() / 256 if c_dtype == torch.bfloat16 else 0)).max()
        assert err < 2e-6 * K ** 0.5 * 4, float(err)


@pytest.mark.parametrize("vocab,d,ff,tokens,seq", [(101, 64, 176, 77, 11), (301, 96, 256, 700, 100), (130, 64, 176, 4100, 820),
                                                   (130, 512, 1376, 6200, 775)])  # of the last some are held back, some not
def test_fp32_training_on_ragged_sizes(vocab, d, ff, tokens, seq):
    """A whole fp32 pass (weight gradients of a block in one launch, residual sums in the products, the embedding's
    gradient with and without the sort) against the same pass on the library's GEMM."""
    m = Llama(vocab=vocab, d=d, n_layers=2, n_heads=d // 32, d_ff=ff, compute_dtype="fp32", seed=8)
    toks = synth.randint(3, tokens + 1, vocab)
    before = blockops.set_gemm_backend(0)
    try:
        want_loss, _ = m.loss_backward(toks[:-1], toks[1:], seq)
        want = m.grads()
        blockops.set_gemm_backend(1)
        for ck in (False, True):
            loss, _ = m.loss_backward(toks[:-1], toks[1:], seq, checkpoint=ck)
            assert abs(loss - want_loss) < 1e-5
            assert rel(m.grads(), want) < 2e-5
    finally:
        blockops.set_gemm_backend(before)
        m.close()


def test_forward_mode_is_refused():
    import torch.autograd.forward_ad as fwd

    q, k, v, tangent = (torch.randn(1, 33, 2, 64, device="cuda") for _ in range(4))
    with fwd.dual_level(), pytest.raises(RuntimeError):
        ops.attention(fwd.make_dual(q, tangent), k, v, 0.125)


def test_two_threads_differentiate_one_graph():
    """Backward passes that share a node take its tensors under the node's lock; one of them releases them at the end."""
    import threading

    q, k, v, d_o = (torch.randn(2, 65, 4, 64, device="cuda", requires_grad=i < 3) for i in range(4))
    o = ops.attention(q, k, v, 0.125)
    want = torch.autograd.grad(o, (q, k, v), d_o, retain_graph=True)
    got, errors = [], []

    def work():
        try:
            for _ in range(20):
                got.append(torch.autograd.grad(o, (q, k, v), d_o, retain_graph=True))
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and len(got) == 80, errors
    assert all(torch.equal(a, b) for g in got for a, b in zip(g, want))
    torch.autograd.grad(o, (q, k, v), d_o)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, (q, k, v), d_o)


# Either side of the lines between chains that are split and those that are not, head sizes between the usual ones: many long
# causal chains of few columns, many short ones of equal length.
@pytest.mark.parametrize("case,dk", [((18, 511, 4, 4, True, 0, 0), 32), ((6, 1446, 4, 2, True, 0, 0), 96), ((36, 114, 4, 2, False, 0, 0), 112),
                                     ((11, 812, 2, 2, True, 22, 0), 80), ((11, 111, 16, 16, True, 20, 16), 80)], ids=str)
def test_lines_between_split_and_unsplit_chains(case, dk):
    B, T, Hq, Hkv, causal, window, sinks = case
    e = errors(*run_attention(B, T, Hq, Hkv, dk, torch.bfloat16, causal, window, sinks))
    assert e[0] < 5e-3 and e[1] < 1e-5 and max(e[2:4]) < 5e-3 and e[4] < 2e-5, e


@pytest.mark.parametrize("grad", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("dk", [64, 128])
@pytest.mark.parametrize("case", [(1, 1, 1, 1, True, 0, 0), (2, 33, 3, 3, False, 0, 0), (3, 300, 5, 5, True, 0, 0), (16, 512, 8, 8, True, 0, 0), (6, 777, 12, 12, False, 0, 0),
                                  (1, 1501, 16, 16, True, 16, 3), (2, 2048, 16, 4, True, 256, 4), (3, 1025, 16, 16, True, 0, 0), (2, 3001, 16, 4, True, 0, 0),
                                  (4, 2000, 16, 16, True, 100, 0), (2, 1000, 16, 4, True, 0, 0), (4, 512, 14, 2, True, 0, 0)], ids=lambda c: "B%d_T%d_H%d_%d_c%d_w%d_s%d" % c)
def test_bf16_rows_of_whole_lines_and_of_others(case, dk, grad):
    """Results whose rows are whole lines of memory and the same results as rows that begin and end inside one, with another's data on either side: the
    same bits, and nothing written beside them. Against float64 as elsewhere: P, dS, O and the gradients rounded to 2 ^ -9 each."""
    B, T, Hq, Hkv, causal, window, sinks = case
    gen = torch.Generator(device="cuda").manual_seed(T + dk)
    draw = lambda h: torch.randn((B, T, h, dk), generator=gen, device="cuda").bfloat16()  # noqa: E731
    q, k, v, d_o = draw(Hq), draw(Hkv), draw(Hkv), draw(Hq)
    scale = float(np.float32(1.0 / np.sqrt(dk)))
    o, lse = ops.attn_fwd(q, k, v, scale, causal, window, sinks)
    got = (o, lse) + ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal, window, sinks, grad_dtype=grad)
    assert max(errors(got, exact_attention(q, k, v, d_o, scale, causal, window, sinks))) < 1e-2
    room = [torch.full((B, T, h, dk + 16), 7.0, device="cuda", dtype=t) for h, t in ((Hq, torch.bfloat16), (Hq, grad), (Hkv, grad), (Hkv, grad))]
    inside = [r[..., 8:-8] for r in room]
    t4, by = ops._t4, ctypes.byref
    _lib.check(_lib.lib().pk_attn_fwd(by(ops._shape(q, k, scale, causal, window, sinks)), by(t4(q)), by(t4(k)), by(t4(v)), by(t4(inside[0])),
                                      ctypes.c_void_p(lse.data_ptr()), ops._stream()))
    ops.attn_bwd(q, k, v, o, lse, d_o, scale, causal, window, sinks, grad,
                 (*inside[1:], torch.empty(ops.bwd_workspace_bytes(q, k, grad, window, sinks), dtype=torch.uint8, device="cuda")))
    for r, i, g in zip(room, inside, (got[0],) + got[2:]):
        assert torch.equal(i, g)
        assert bool((r[..., :8] == 7.0).all()) and bool((r[..., -8:] == 7.0).all())


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("vocab,d,ff,tokens,chunk,fused", [(130, 64, 176, 64, 0, True), (37, 12, 20, 30, 7, True), (1001, 256, 700, 700, 256, True),
                                                           (5, 8, 10, 3, 0, True), (504, 512, 1376, 4100, 0, True), (130, 64, 176, 64, 0, False)])
def test_nothing_is_left_of_the_gradients_before(dtype, vocab, d, ff, tokens, chunk, fused):
    """A pass on a model whose last pass left NaN in every gradient, with and without a pass forward alone between them, against the same pass
    on a new model: the head's product writes the embedding's gradient where it is the first to, whole and beside words that no token has."""
    toks = [synth.randint(s, tokens + 1, vocab) for s in (3, 4)]

    def new():
        m = Llama(vocab=vocab, d=d, n_layers=1, n_heads=2, d_ff=ff, compute_dtype=dtype, seed=8)
        if chunk:
            m.set_head_chunk(chunk)
        return m

    m, other = new(), new()
    params = other.params()
    other.loss_backward(toks[1][:-1], toks[1][1:], 0, fused_head=fused)
    want = other.grads()
    other.close()
    for forward_between in (False, True):
        m.set_params({k: np.full_like(v, np.nan) for k, v in params.items()})
        m.loss_backward(toks[0][:-1], toks[0][1:], 0, fused_head=fused)
        assert all(np.isnan(g).any() for g in m.grads().values())
        m.set_params(params)
        if forward_between:
            m.loss_backward(toks[0][:-1], toks[0][1:], 0, backward=False, fused_head=fused)
            assert all((g == 0).all() for g in m.grads().values())
        m.loss_backward(toks[1][:-1], toks[1][1:], 0, fused_head=fused)
        for k, g in m.grads().items():
            assert np.array_equal(g, want[k]), k
    m.close()


@pytest.mark.parametrize("n,vocab,d", [(1, 3, 5), (3, 1, 700), (1023, 40, 33), (4097, 5000, 64), (8191, 32000, 513), (8192, 7, 130), (8192, 1, 1025), (8193, 300, 64),
                                       (4097, 3, 1024), (4097, 2, 1025), (4095, 3, 1300), (8190, 4, 1024), (257, 40, 700)])
def test_embedding_gradient_of_ids_looked_through(n, vocab, d):
    """Up to 8192 ids are looked through by every workgroup, four to a load: counts that are no multiple of four, one beside the sort's, ids that all
    rows share or none, columns short of one and of two a thread and beside the sort's, and ids that do not begin on 16 bytes. A row's sum is formed in row order: the bits
    of the same additions one after the other."""
    rng = np.random.RandomState(n + d)
    ids, dy = rng.randint(0, vocab, n).astype(np.int32), rng.randn(n, d).astype(np.float32)
    want = np.zeros((vocab, d), np.float32)
    for i in range(n):
        want[ids[i]] += dy[i]
    for skip in (0, 1):
        there = torch.zeros(n + skip, dtype=torch.int32, device="cuda")
        there[skip:] = torch.from_numpy(ids).cuda()
        got = blockops.embedding(torch.zeros((vocab, d), device="cuda"), there[skip:], torch.from_numpy(dy).cuda())[1]
        assert np.array_equal(got.cpu().numpy(), want)
