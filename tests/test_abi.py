"""The C-ABI library loads and exports every symbol include/paperkiln_amd.h declares. No GPU, no compute."""
import ctypes
import os
import re

import pytest

from paperkiln_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    text = open(os.path.join(ROOT, "include", "paperkiln_amd.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(pk_[a-z0-9_]+)\s*\(", text)))


def test_header_and_binding_agree():
    assert declared_symbols() == sorted(_lib.EXPORTS)


def test_library_exports_every_declared_symbol():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail(f"{_lib.LIB_PATH} not built: run __graft_entry__.build()")
    L = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared_symbols():
        assert hasattr(L, name), name


def test_argument_errors_do_not_need_a_gpu():
    """Shape/argument validation happens before any HIP call and mirrors the reference's throws."""
    L = _lib.lib()
    sh = _lib.AttnShape(1, 8, 3, 2, 4, 1, 0, 0, 0.5, _lib.PK_F32, _lib.PK_F32)  # Hq % Hkv != 0
    t = _lib.Tensor4(0, 0, 0, 0)
    rc = L.pk_attn_fwd(ctypes.byref(sh), ctypes.byref(t), ctypes.byref(t), ctypes.byref(t), ctypes.byref(t), None, None)
    assert rc == 1 and b"shape mismatch" in L.pk_last_error()
    sh = _lib.AttnShape(1, 8, 2, 2, 4, 0, 3, 0, 0.5, _lib.PK_F32, _lib.PK_F32)  # window without causal
    assert L.pk_attn_fwd(ctypes.byref(sh), ctypes.byref(t), ctypes.byref(t), ctypes.byref(t), ctypes.byref(t), None, None) == 2
    sh = _lib.AttnShape(1, 8, 2, 2, 4, 1, 0, 0, 0.5, _lib.PK_F32, _lib.PK_F32)
    assert L.pk_attn_fwd(ctypes.byref(sh), ctypes.byref(t), ctypes.byref(t), ctypes.byref(t), ctypes.byref(t), None, None) == 2  # null tensors
    assert L.pk_attn_bwd_workspace_bytes(ctypes.byref(sh)) == 4 * 1 * 2 * 8


def test_backward_workspace_follows_the_mask():
    """pk_attn_bwd_workspace_bytes: delta [B, Hq, T] fp32 for every mask; query heads that share KV heads add the
    per-split partial dK / dV where the kernel of that launch deals them to several workgroups; a band mask with 1..32 sink keys on a
    sequence longer than key block 0's band adds the partial sink rows of a split sink tail
    ((chunks of 512 queries + 1) x {dK, dV} x 32 rows x head_dim fp32 per (batch, KV head), 256-byte aligned)."""
    L = _lib.lib()
    B, T, Hq, Hkv, dk = 2, 4096, 8, 4, 128
    delta = 4 * B * Hq * T

    def ws(window, sinks, t=T):
        sh = _lib.AttnShape(B, t, Hq, Hkv, dk, 1, window, sinks, 0.5, _lib.PK_BF16, _lib.PK_BF16)
        return L.pk_attn_bwd_workspace_bytes(ctypes.byref(sh))

    # no band, 2 query heads per KV head, 16 paired key blocks x 8 (batch, KV head) units = 128 dK/dV workgroups for
    # 256 CUs: the heads of a group are dealt to 2 workgroups, whose fp32 partial dK and dV follow delta
    assert ws(0, 0) == delta + 4 * 2 * (B * Hkv) * 2 * T * dk
    mha = _lib.AttnShape(B, T, Hq, Hq, dk, 1, 0, 0, 0.5, _lib.PK_BF16, _lib.PK_BF16)
    assert L.pk_attn_bwd_workspace_bytes(ctypes.byref(mha)) == delta   # one query head per KV head: nothing to deal
    assert ws(256, 0) == delta          # no sink keys: nothing to split
    assert ws(256, 33) == delta         # more sink keys than one wavefront owns: not split
    q0 = ((127 + 256 - 1) // 64 + 1) * 64   # first 64-query tile wholly past key block 0's band
    nch = -(-(T - q0) // 512)
    assert ws(256, 4) == delta + 4 * B * Hkv * (nch + 1) * 2 * 32 * dk
    assert ws(256, 4, t=q0) == 4 * B * Hq * q0   # the sequence ends with the band: no tail
    odd = 4 * B * Hq * 4001                      # delta not a multiple of 256 bytes: the tail starts aligned
    assert ws(256, 4, t=4001) == odd + (256 - odd % 256) % 256 + 4 * B * Hkv * (-(-(4001 - q0) // 512) + 1) * 2 * 32 * dk


def test_partial_sums_are_asked_for_where_a_kernel_writes_them():
    """Query heads that share KV heads: fp32 partial dK / dV are part of the workspace only where the dK/dV launch goes to
    a kernel that deals a group's heads to several workgroups; scale and gradient type do not change the answer."""
    L = _lib.lib()

    def ws(B, T, Hq, Hkv, dk, dtype, causal=1, window=0, scale=0.5, grad=_lib.PK_F32):
        sh = _lib.AttnShape(B, T, Hq, Hkv, dk, causal, window, 0, scale, dtype, grad)
        return L.pk_attn_bwd_workspace_bytes(ctypes.byref(sh)) - 4 * B * Hq * T

    f32, bf16 = _lib.PK_F32, _lib.PK_BF16
    assert ws(4, 4096, 16, 4, 128, f32) == 0     # walked in one workgroup by the 128-key kernel (134 MB otherwise)
    assert ws(31, 256, 16, 4, 64, bf16) == 0     # by the 32-key kernel (65 MB otherwise)
    assert ws(1, 700, 14, 2, 256, bf16) == 0     # head sizes of the scalar kernels
    parts = 4 * 2 * 2 * 4096 * 128 * 16
    assert ws(4, 4096, 16, 4, 128, bf16) == parts  # 2 splits of 16 units: the 64-key kernel
    for scale, grad in ((-1.0, f32), (0.0, bf16)):
        assert ws(4, 4096, 16, 4, 128, bf16, scale=scale, grad=grad) == parts
    assert ws(1, 256, 14, 2, 64, f32) > 0 and ws(1, 256, 14, 2, 80, bf16, window=64) > 0  # kernels that split the queries


def test_workspace_of_the_torch_front_end_fits_both_masks():
    """ops.bwd_workspace_bytes is not told whether the mask is causal: it has to be enough for either."""
    import random

    import torch

    from paperkiln_amd import ops
    L, rng = _lib.lib(), random.Random(5)
    for _ in range(400):
        dtype = rng.choice([torch.float32, torch.bfloat16])
        B, Hkv, rep, dk = rng.randint(1, 40), rng.randint(1, 4), rng.randint(1, 8), rng.choice([32, 64, 80, 128])
        T = int(2 ** rng.uniform(0, 13))
        q, k = (torch.empty((B, T, h, dk), dtype=dtype, device="meta") for h in (Hkv * rep, Hkv))
        code = _lib.PK_F32 if dtype == torch.float32 else _lib.PK_BF16
        for causal in (0, 1):
            sh = _lib.AttnShape(B, T, Hkv * rep, Hkv, dk, causal, 0, 0, 0.3, code, code)
            assert ops.bwd_workspace_bytes(q, k) >= L.pk_attn_bwd_workspace_bytes(ctypes.byref(sh))


def test_a_window_that_covers_the_sequence_is_no_band():
    """The reference takes size_t window / sinks and defines window >= seq_len as plain causal attention
    (tests/test_swa.cpp:47-57), so INT32_MAX is a legal "no band": the shape is brought into range on the host,
    before any index arithmetic, and sizes its workspace as the causal mask does."""
    L = _lib.lib()
    B, T, Hq, Hkv, dk = 2, 4096, 8, 8, 128

    def ws(window, sinks):
        sh = _lib.AttnShape(B, T, Hq, Hkv, dk, 1, window, sinks, 0.5, _lib.PK_BF16, _lib.PK_BF16)
        return L.pk_attn_bwd_workspace_bytes(ctypes.byref(sh))

    causal = ws(0, 0)
    assert causal == 4 * B * Hq * T
    for window in (T, T + 1, 2**31 - 1):
        for sinks in (0, 4, 2**31 - 1):
            assert ws(window, sinks) == causal
    assert ws(T // 2, 4) > causal         # a real band with sink keys still gets its sink-tail rows
    assert ws(256, 2**31 - 1) == causal   # more sink keys than tokens: every key is a sink, nothing to split
    sh = _lib.AttnShape(1, 2**24 + 1, 1, 1, 64, 1, 0, 0, 0.5, _lib.PK_BF16, _lib.PK_BF16)
    assert L.pk_attn_bwd_workspace_bytes(ctypes.byref(sh)) == 0 and b"2^24" in L.pk_last_error()


def test_handle_and_pointer_errors_do_not_need_a_gpu():
    """A NULL model handle and a pointer pk_alloc never returned are reported, not dereferenced or ignored."""
    L = _lib.lib()
    r, c = ctypes.c_int64(), ctypes.c_int64()
    assert L.pk_llama_param_info(None, 0, None, 0, ctypes.byref(r), ctypes.byref(c)) == 2
    assert b"null model handle" in L.pk_last_error()
    assert L.pk_llama_num_params(None) == -1
    assert L.pk_llama_adamw_step(None, 1e-3, 0.9, 0.999, 1e-8, 0.0, 0.0, None) == 2
    assert L.pk_llama_set_head_chunk(None, 128) == 2
    assert L.pk_llama_destroy(None) == 0
    buf = ctypes.create_string_buffer(64)
    assert L.pk_free(ctypes.cast(buf, ctypes.c_void_p)) == 2 and b"pk_alloc" in L.pk_last_error()
    assert L.pk_free(None) == 0
    assert L.pk_alloc(64, None) == 2


# (B, T, Hq, Hkv, head_dim, causal, window, sinks); what is apart measured 1.03 to 1.8 times as slow in one launch
BWD_FORMS = ("APART", "SPLIT", "SPLIT_JOINED", "JOINED", "F32_SPLIT", "F32_PARTS", "F32_PARTS_ALL")
BF16_LAUNCHES = [
    ("JOINED", (4, 307, 16, 8, 128, 1, 0, 0)), ("JOINED", (4, 559, 8, 8, 128, 1, 71, 0)), ("SPLIT_JOINED", (8, 470, 8, 8, 64, 1, 0, 0)),
    ("SPLIT_JOINED", (58, 148, 2, 2, 48, 1, 0, 0)), ("SPLIT_JOINED", (7, 393, 14, 2, 96, 1, 0, 0)), ("SPLIT", (1, 128, 4, 4, 64, 1, 0, 0)),
    # groups of heads that are not dealt out under a band, few blocks, a tail of sinks beside few, a second round of the chip
    ("APART", (1, 3396, 7, 1, 128, 1, 477, 0)), ("APART", (2, 372, 16, 4, 128, 1, 219, 0)), ("SPLIT", (1, 1702, 2, 2, 128, 1, 73, 0)),
    ("APART", (1, 697, 8, 8, 128, 1, 181, 4)), ("APART", (1, 3220, 8, 8, 128, 1, 305, 0)), ("APART", (1, 2006, 4, 4, 128, 0, 0, 0)),
    ("APART", (99, 44, 4, 2, 128, 1, 0, 0)), ("APART", (1, 3810, 8, 8, 32, 1, 1771, 0)), ("APART", (1, 4433, 8, 4, 64, 0, 0, 0)),
    ("APART", (1, 4950, 8, 8, 64, 1, 25, 0)), ("APART", (1, 3156, 16, 4, 96, 0, 0, 0)), ("APART", (53, 222, 4, 4, 96, 0, 0, 0))]
F32_LAUNCHES = [
    ("F32_PARTS", (4, 1024, 8, 8, 64, 1, 0, 0)), ("F32_PARTS_ALL", (4, 313, 16, 16, 64, 1, 0, 0)), ("F32_PARTS_ALL", (1, 4576, 1, 1, 128, 1, 0, 0)),
    ("F32_SPLIT", (2, 128, 4, 4, 32, 1, 0, 0)), ("APART", (4, 4096, 16, 16, 128, 1, 0, 0)), ("F32_PARTS_ALL", (2, 3300, 1, 1, 80, 1, 0, 0)),
    ("APART", (1, 3183, 8, 2, 64, 0, 0, 0)), ("APART", (3, 4549, 2, 2, 64, 0, 0, 0)), ("APART", (1, 3353, 8, 4, 32, 0, 0, 0)),
    ("APART", (51, 87, 4, 1, 128, 1, 0, 0)), ("APART", (99, 44, 2, 2, 96, 0, 0, 0)), ("APART", (1, 654, 8, 8, 80, 1, 180, 16)),
    ("F32_SPLIT", (3, 137, 16, 16, 32, 1, 27, 16)), ("F32_SPLIT", (1, 4127, 2, 2, 32, 1, 966, 0)), ("APART", (1, 3220, 8, 8, 96, 1, 305, 0))]


@pytest.mark.parametrize("dtype,form,shape", [(_lib.PK_BF16, *x) for x in BF16_LAUNCHES] + [(_lib.PK_F32, *x) for x in F32_LAUNCHES], ids=str)
def test_which_launches_a_whole_backward_takes(dtype, form, shape):
    """dQ and dK/dV go into one launch where that is ahead of two, or of the blocks of 32 rows that share one as well."""
    assert BWD_FORMS[_lib.lib().pk_bwd_of_shape(ctypes.byref(_lib.AttnShape(*shape, 1.0, dtype, dtype)))] == form


@pytest.mark.parametrize("n,d,scans", [(1, 64, 1), (4096, 1024, 1), (4096, 4096, 1), (4097, 512, 1), (4097, 1024, 1), (4097, 1025, 0), (8192, 512, 1), (8192, 1024, 1),
                                       (8192, 2048, 0), (8193, 64, 0), (1 << 20, 512, 0)])
def test_which_embedding_gradients_go_without_the_sort(n, d, scans):
    """Workgroups that look through all ids and take a row's columns 512 at a time: as far as they are ahead of the sort, in ids and in columns."""
    assert _lib.lib().pk_embedding_scans(ctypes.c_int64(n), ctypes.c_int64(d)) == scans
