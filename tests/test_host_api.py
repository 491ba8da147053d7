"""CPU-side tests: the C-ABI library loads and exports what include/flash_attn_gfx950.h declares, argument
validation returns errors instead of aborting, the seqlen rounding follows fmha_api.cpp, and the pure-host helpers
(bert_padding, convert_blockmask, rotary) match their specifications.  Nothing here launches a kernel."""
import ctypes
import inspect
import os
import re

import numpy as np
import pytest
import torch

from oracle import attention_oracle as orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol(lib):
    header = open(os.path.join(ROOT, "include", "flash_attn_gfx950.h")).read()
    declared = set(re.findall(r"^\s*(?:int|size_t|void|uint64_t|const char\*)\s+(fa_\w+)\s*\(", header, re.M))
    from flash_attn import flash_attn_gfx950 as be
    assert declared == set(be.EXPORTED_SYMBOLS)
    # the instrumentation entry point of bench.py has a header of its own and is not part of the drop-in boundary
    bench = open(os.path.join(ROOT, "include", "flash_attn_gfx950_bench.h")).read()
    declared_bench = set(re.findall(r"^\s*(?:int|size_t|void)\s+(fa_\w+)\s*\(", bench, re.M))
    assert declared_bench == set(be.BENCH_SYMBOLS) and not (declared & declared_bench)
    for name in declared | declared_bench:
        assert hasattr(lib, name), name
    assert lib.fa_abi_version() == be.FA_ABI_VERSION == 5


@pytest.mark.parametrize("version, says", [(4, "has ABI version 4, binding expects 5"), (5, "lacks fa_fwd, .*fa_token_positions.*build it again"),
                                           (None, "has no fa_abi_version")])
def test_another_library_is_named_as_such(lib, tmp_path, monkeypatch, version, says):
    """a library of another version, or one built before an entry point was added, is refused with a message, not by a missing symbol; the one in
    use stays in use"""
    import subprocess
    from flash_attn import flash_attn_gfx950 as be
    src, so = tmp_path / "other.c", tmp_path / "other.so"
    src.write_text("int nothing;" if version is None else "int fa_abi_version(void) { return %d; }" % version)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    for name, value in (("_lib", None), ("_host", None), ("_passes", None), ("LIB_PATH", str(so))):
        monkeypatch.setattr(be, name, value)
    with pytest.raises(RuntimeError, match=says):
        be.load_library()
    assert be._lib is None and be._host is None
    monkeypatch.undo()
    assert be.load_library() is lib


def test_struct_layout_matches_library(lib):
    """a wrong struct size is reported as an ABI mismatch; the right size passes that check"""
    from flash_attn import flash_attn_gfx950 as be
    a = be.FwdArgs()
    a.struct_bytes = ctypes.sizeof(a) - 8
    assert lib.fa_fwd(ctypes.byref(a)) == -1 and b"ABI mismatch" in lib.fa_last_error()
    a.struct_bytes = ctypes.sizeof(a)
    a.dtype = 7
    assert lib.fa_fwd(ctypes.byref(a)) == -1 and b"dtype" in lib.fa_last_error()
    g = be.BwdArgs()
    g.struct_bytes = ctypes.sizeof(g)
    g.dtype = 7
    assert lib.fa_bwd(ctypes.byref(g)) == -1 and b"dtype" in lib.fa_last_error()


def _valid_fwd_args(be):
    a = be.FwdArgs()
    a.struct_bytes = ctypes.sizeof(a)
    a.dtype = be.FA_FP16
    a.batch, a.nheads, a.head_dim = 1, 1, 64
    a.total_q = a.total_k = 16
    a.max_seqlen_q = a.max_seqlen_k = 16
    a.p_dropout, a.softmax_scale = 0.0, 0.125
    for f in ("q_row_stride", "k_row_stride", "v_row_stride", "o_row_stride"):
        setattr(a, f, 64)
    for f in ("q_head_stride", "k_head_stride", "v_head_stride", "o_head_stride"):
        setattr(a, f, 64)
    return a


@pytest.mark.parametrize("field,value,needle", [
    ("batch", 0, b"batch_size"),                 # fmha_api.cpp:223
    ("head_dim", 48, b"head_size"),              # :224
    ("p_dropout", 1.0, b"p_dropout"),            # :113
    ("p_dropout", -0.1, b"p_dropout"),
    ("softmax_scale", 0.0, b"softmax_scale"),
    ("max_seqlen_q", 0, b"max_seqlen"),
])
def test_forward_argument_checks(lib, field, value, needle):
    from flash_attn import flash_attn_gfx950 as be
    a = _valid_fwd_args(be)
    setattr(a, field, value)
    rc = lib.fa_fwd(ctypes.byref(a))
    assert rc == -1 and needle in lib.fa_last_error(), lib.fa_last_error()


def test_null_pointers_and_alignment_are_errors_not_crashes(lib):
    from flash_attn import flash_attn_gfx950 as be
    a = _valid_fwd_args(be)
    assert lib.fa_fwd(ctypes.byref(a)) == -1 and b"NULL" in lib.fa_last_error()
    for f in ("q", "k", "v", "o", "softmax_lse", "cu_seqlens_q", "cu_seqlens_k"):
        setattr(a, f, 0x1000)
    a.q = 0x1008
    assert lib.fa_fwd(ctypes.byref(a)) == -1 and b"aligned" in lib.fa_last_error()
    a.q = 0x1000
    a.k_row_stride = 70
    assert lib.fa_fwd(ctypes.byref(a)) == -1 and b"strides" in lib.fa_last_error()
    a.k_row_stride = 64
    a.blockmask = 0x1000  # dense entry point refuses a blockmask, block entry point refuses its absence
    assert lib.fa_fwd(ctypes.byref(a)) == -1 and b"blockmask" in lib.fa_last_error()
    a.blockmask = None
    assert lib.fa_fwd_block(ctypes.byref(a)) == -1 and b"blockmask" in lib.fa_last_error()
    assert lib.fa_fwd(None) == -1


@pytest.mark.parametrize("max_q", [1, 100])  # decode kernel, forward kernel
@pytest.mark.parametrize("keys", [100, 4096])
@pytest.mark.parametrize("field,value", [("batch", 0), ("nheads", 0), ("max_seqlen_q", 0), ("max_seqlen_k", 0), ("max_seqlen_k", -1),
                                         ("batch", -1), ("nheads", -1)])
def test_size_queries_of_calls_that_are_refused(lib, field, value, keys, max_q):
    """The callers ask for the scratch before the call checks its arguments (an empty cache, an empty batch): the queries answer
    0 and the call returns its error."""
    from flash_attn import flash_attn_gfx950 as be
    a = _valid_fwd_args(be)
    a.max_seqlen_q, a.max_seqlen_k = max_q, keys
    setattr(a, field, value)
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) == 0
    assert lib.fa_fwd(ctypes.byref(a)) == -1 and b"must be positive" in lib.fa_last_error()
    g = be.BwdArgs()
    g.struct_bytes = ctypes.sizeof(g)
    g.batch, g.nheads, g.head_dim, g.total_q, g.total_k, g.max_seqlen_q, g.max_seqlen_k = 1, 2, 64, 100, 5000, max_q, keys
    g.softmax_scale = 0.125
    setattr(g, field, value)
    assert lib.fa_bwd_workspace_bytes(ctypes.byref(g)) == 0
    assert lib.fa_bwd(ctypes.byref(g)) == -1 and b"must be positive" in lib.fa_last_error()


def test_block_sparse_needs_workspace_also_when_causal(lib):
    from flash_attn import flash_attn_gfx950 as be
    a = _valid_fwd_args(be)
    for f in ("q", "k", "v", "o", "softmax_lse", "cu_seqlens_q", "cu_seqlens_k", "blockmask"):
        setattr(a, f, 0x1000)
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) > 0
    assert lib.fa_fwd_block(ctypes.byref(a)) == -2 and b"workspace" in lib.fa_last_error()
    a.is_causal = 1  # accepted together with a blockmask: the same workspace rule applies
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) > 0
    assert lib.fa_fwd_block(ctypes.byref(a)) == -2 and b"workspace" in lib.fa_last_error()


def test_workspace_sizes(lib):
    from flash_attn import flash_attn_gfx950 as be
    a = _valid_fwd_args(be)
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) == 0  # the dense forward needs no scratch (no o_tmp)
    g = be.BwdArgs()
    g.struct_bytes = ctypes.sizeof(g)
    g.batch, g.nheads, g.head_dim, g.total_q, g.total_k = 2, 3, 64, 100, 100
    g.max_seqlen_q = g.max_seqlen_k = 64
    assert lib.fa_bwd_workspace_bytes(ctypes.byref(g)) == 0  # nor the dense backward (no fp32 dq_tmp)
    g.blockmask = 0x1000
    assert lib.fa_bwd_workspace_bytes(ctypes.byref(g)) > 0   # block-sparse: room for the block activity maps
    # dropout keep words: one bit per (batch, head, query, key), both lengths rounded up to 128
    assert lib.fa_keep_words_bytes(8, 12, 512, 512) == 8 * 12 * 512 * 512 // 8
    assert lib.fa_keep_words_bytes(1, 1, 100, 300) == 128 * 384 // 8
    assert lib.fa_keep_words_bytes(2, 3, 129, 1) == 2 * 3 * 256 * 128 // 8
    assert lib.fa_keep_words_bytes(0, 3, 129, 1) == 0 and lib.fa_keep_words_bytes(2, 3, 0, 1) == 0


@pytest.mark.parametrize("d,sq,sk,sparse,want", [
    (64, 1, 1, False, (16, 128)),          # fmha_api.cpp:235-236
    (64, 128, 129, False, (128, 256)),     # :237-238
    (64, 500, 500, False, (512, 512)),     # :234 with blocksize_c = 256
    (64, 513, 513, False, (528, 768)),
    (128, 300, 300, False, (304, 384)),    # blocksize_c = 128 for head_size 128 off sm80 (:232)
    (32, 100, 100, True, (112, 256)),      # :509-513
    (64, 4096, 4096, True, (4096, 4096)),
    (64, 4097, 4097, True, (4112, 4352)),
])
def test_round_seqlens(lib, d, sq, sk, sparse, want):
    from flash_attn import flash_attn_gfx950 as be
    assert be.round_seqlens(d, sq, sk, sparse) == want


def test_python_checks_raise_runtime_error():
    """the binding's own checks mirror TORCH_CHECK -> RuntimeError before anything touches a GPU"""
    from flash_attn import flash_attn_gfx950 as be
    q = torch.zeros(16, 1, 64, dtype=torch.float32)
    cu = torch.tensor([0, 16], dtype=torch.int32)
    with pytest.raises(RuntimeError, match="fp16 or bf16"):
        be.fwd(q, q, q, cu, cu, 16, 16, 0.0, 0.125, False, False, False, None)
    h = q.half()
    with pytest.raises(RuntimeError, match="GPU"):
        be.fwd(h, h, h, cu, cu, 16, 16, 0.0, 0.125, False, False, False, None)
    with pytest.raises(RuntimeError, match="head_size"):
        be.fwd(h[..., :48], h[..., :48], h[..., :48], cu, cu, 16, 16, 0.0, 0.125, False, False, False, None)


def test_public_signatures_match_the_reference():
    """names, order and defaults of flash_attn_interface.py:151-252 and flash_blocksparse_attn_interface.py:135-137"""
    from flash_attn import flash_attn_interface as fi
    from flash_attn import flash_blocksparse_attn_interface as bi
    from flash_attn import bert_padding as bp

    def sig(f):
        return [(n, p.default if p.default is not inspect.Parameter.empty else "<req>")
                for n, p in inspect.signature(f).parameters.items()]

    # the functions that reach the kernels take the reference's parameters followed by two extensions,
    # alibi_slopes=None and attn_bias=None (attention bias: planned in the reference's README, absent from its API)
    ext = [("alibi_slopes", None), ("attn_bias", None)]
    assert sig(fi.flash_attn_unpadded_qkvpacked_func) == [
        ("qkv", "<req>"), ("cu_seqlens", "<req>"), ("max_seqlen", "<req>"), ("dropout_p", "<req>"),
        ("softmax_scale", None), ("causal", False), ("return_attn_probs", False)] + ext
    assert sig(fi.flash_attn_unpadded_kvpacked_func) == [
        ("q", "<req>"), ("kv", "<req>"), ("cu_seqlens_q", "<req>"), ("cu_seqlens_k", "<req>"),
        ("max_seqlen_q", "<req>"), ("max_seqlen_k", "<req>"), ("dropout_p", "<req>"), ("softmax_scale", None),
        ("causal", False), ("return_attn_probs", False)] + ext
    assert sig(fi.flash_attn_unpadded_func) == [
        ("q", "<req>"), ("k", "<req>"), ("v", "<req>"), ("cu_seqlens_q", "<req>"), ("cu_seqlens_k", "<req>"),
        ("max_seqlen_q", "<req>"), ("max_seqlen_k", "<req>"), ("dropout_p", "<req>"), ("softmax_scale", None),
        ("causal", False), ("return_attn_probs", False)] + ext
    assert sig(fi.flash_attn_func) == [
        ("qkv", "<req>"), ("cu_seqlens", "<req>"), ("dropout_p", "<req>"), ("max_s", "<req>"),
        ("softmax_scale", None), ("causal", False), ("return_attn_probs", False)]
    assert sig(bi.flash_blocksparse_attn_func) == [
        ("qkv", "<req>"), ("cu_seqlens", "<req>"), ("blockmask", "<req>"), ("dropout_p", "<req>"), ("max_s", "<req>"),
        ("softmax_scale", None), ("causal", False), ("return_attn_probs", False), ("convert_mask", True)] + ext
    assert [n for n, _ in sig(bp.unpad_input)] == ["hidden_states", "attention_mask"]
    assert [n for n, _ in sig(bp.pad_input)] == ["hidden_states", "indices", "batch", "seqlen"]
    for cls in ("FlashAttnQKVPackedFunc", "FlashAttnKVPackedFunc", "FlashAttnFunc"):
        assert issubclass(getattr(fi, cls), torch.autograd.Function)
    from flash_attn import flash_attn_gfx950 as be
    assert list(inspect.signature(be.fwd).parameters) == [
        "q", "k", "v", "cu_seqlens_q", "cu_seqlens_k", "max_seqlen_q", "max_seqlen_k", "p_dropout", "softmax_scale",
        "zero_tensors", "is_causal", "return_softmax", "gen", "alibi_slopes", "keep_words", "attn_bias", "rotary",
        "q_rot"]  # fmha_api.cpp:173-186 + extensions
    assert sig(fi.flash_attn_unpadded_qkvpacked_rotary_func) == [
        ("qkv", "<req>"), ("cos_half", "<req>"), ("sin_half", "<req>"), ("cu_seqlens", "<req>"), ("max_seqlen", "<req>"),
        ("dropout_p", "<req>"), ("softmax_scale", None), ("causal", False)]  # extension: rotary embedding inside the kernels
    assert list(inspect.signature(be.bwd_block).parameters) == [
        "dout", "q", "k", "v", "out", "softmax_lse", "dq", "dk", "dv", "cu_seqlens_q", "cu_seqlens_k", "blockmask",
        "max_seqlen_q", "max_seqlen_k", "p_dropout", "softmax_scale", "is_causal", "gen", "row_order", "alibi_slopes",
        "attn_bias", "dbias"]  # fmha_api.cpp:575-594 + extensions


def test_blockmask_row_order_is_a_permutation_that_groups_similar_rows():
    """fa_blocksparse_row_order (host code of the library) lists every row block once, is deterministic, never stages more
    key blocks than the plain order, saves a third of the staged blocks and a fifth of the waves' work on independently drawn
    16 x 256 blocks, handles more than 64 key blocks and ragged ends, and leaves layouts made of whole 128-row tiles alone"""
    from flash_attn import flash_attn_gfx950 as be
    g = torch.Generator().manual_seed(0)

    def staged(m, order):  # key blocks a workgroup (eight consecutive entries) has to stage, summed
        return sum(int(m[order[i:i + 8]].any(0).sum()) for i in range(0, len(order), 8))

    def computed(m, order):  # key blocks a wave (two consecutive entries) has to compute on, summed
        return sum(int(m[order[i:i + 2]].any(0).sum()) for i in range(0, len(order), 2))

    for nrow, ncol, dens in ((256, 16, 0.25), (19, 2, 0.5), (64, 4, 0.1), (8, 1, 1.0), (1, 1, 0.0), (100, 70, 0.2)):
        m = torch.rand(nrow, ncol, generator=g) < dens
        order = be.blockmask_row_order(m)
        assert order.dtype == torch.int32 and sorted(order.tolist()) == list(range(nrow))
        assert torch.equal(order, be.blockmask_row_order(m))
        ident = torch.arange(nrow)
        assert staged(m, order.long()) <= staged(m, ident)
        if nrow == 256:
            assert staged(m, order.long()) < 0.7 * staged(m, ident)
            assert computed(m, order.long()) < 0.82 * computed(m, ident)
    tiles = (torch.rand(16, 16, generator=g) < 0.3).repeat_interleave(16, 0)  # 256 x 256 blocks
    assert be.blockmask_row_order(tiles).tolist() == list(range(256))
    lib = be.load_library()
    assert lib.fa_blocksparse_row_order(None, 4, 4, None) == -1


@pytest.mark.parametrize("rows, cols, crc", [(256, 16, 501783833), (37, 5, 137879411), (1, 1, 558161692), (100, 64, 4146698765), (130, 70, 3019294916)])
def test_blockmask_row_order_stays_what_it_was(rows, cols, crc):
    """The order of a layout, which results follow in their last bits, is the one that recomputing every group's lists at every exchange gives (checksums
    of its orders): whole and partial groups, one row, one word of key blocks and two"""
    import zlib
    from flash_attn import flash_attn_gfx950 as be
    r, c = torch.arange(rows)[:, None], torch.arange(cols)[None]
    layout = ((r * 7 + c * 13) * (r + 3 * c + 1) + r * r // 5) % 11 < 4
    assert zlib.crc32(be.blockmask_row_order(layout).numpy().tobytes()) == crc


# ---------------------------------------------------------------- host helpers
def _layouts_to_order(n):
    """0 / 1 layouts whose row orders are not the plain one and differ"""
    g = torch.Generator().manual_seed(3)
    return [torch.rand(64, 16, generator=g) < 0.3 for _ in range(n)]


def test_row_order_follows_the_masks_values_not_its_address():
    """A converted mask at the address of one that is gone, with the same shape and version, has its own order; so does a mask after a write to it."""
    from flash_attn import flash_attn_gfx950 as be, flash_blocksparse_attn_interface as bi
    a, b, c = _layouts_to_order(3)
    want = [be.blockmask_row_order(m) for m in (a, b, c)]
    assert not torch.equal(want[0], want[1]) and not torch.equal(want[1], want[2])
    memory = np.empty((16, 64), dtype=np.int32)
    at = None
    for m, order in ((a, want[0]), (b, want[1])):
        memory[:] = bi.convert_blockmask(m, causal=False).numpy()
        conv = torch.from_numpy(memory)
        assert at in (None, conv.data_ptr()) and conv._version == 0
        at = conv.data_ptr()
        assert torch.equal(bi._row_order(conv, False), order)
        del conv
    conv = bi.convert_blockmask(b, causal=False)
    assert torch.equal(bi._row_order(conv, False), want[1])
    conv.copy_(bi.convert_blockmask(c, causal=False))
    assert torch.equal(bi._row_order(conv, False), want[2])
    assert bi._row_order(conv, True) is None


def test_row_order_is_worked_out_once_per_mask(monkeypatch):
    """Kept with the caller's layout (whose converted form is a new tensor in every call), with views of it, and by its values where a call
    makes a new layout; nothing is kept for a layout that is gone but the last 64 values."""
    import gc
    from flash_attn import flash_attn_gfx950 as be, flash_blocksparse_attn_interface as bi
    calls, reads = [], []
    worked_out, read = be.blockmask_row_order, bi._row_order_of_values
    monkeypatch.setattr(be, "blockmask_row_order", lambda m: calls.append(1) or worked_out(m))
    monkeypatch.setattr(bi, "_row_order_of_values", lambda m: reads.append(1) or read(m))
    bi._ORDERS_OF_CONTENTS.clear()
    gc.collect()
    kept = len(bi._ORDERS_OF_MASKS)
    layout, = _layouts_to_order(1)

    def order(m):
        return bi._row_order(bi.convert_blockmask(m, causal=False), False, m)

    first = order(layout)
    assert all(order(layout) is first for _ in range(3)) and (len(calls), len(reads)) == (1, 1)
    part = order(layout[:32, :8])
    assert order(layout[:32, :8]) is part and part.numel() == 32 and (len(calls), len(reads)) == (2, 2)
    assert torch.equal(order(layout.clone()), first) and (len(calls), len(reads)) == (2, 3)
    with torch.inference_mode():
        assert order(layout) is first and order(layout[:32, :8]) is part and len(reads) == 3
        assert torch.equal(order(layout.clone()), first) and len(calls) == 2 and len(reads) == 4  # (an inference tensor has no version)
    layout[0] = ~layout[0]
    assert not torch.equal(order(layout), first) and len(calls) == 3
    for i in range(70):
        order(torch.rand(16, 4, generator=torch.Generator().manual_seed(i)) < 0.5)
    assert len(bi._ORDERS_OF_CONTENTS) <= 64
    del layout
    gc.collect()
    assert len(bi._ORDERS_OF_MASKS) == kept


def test_convert_blockmask_matches_spec():
    from flash_attn.flash_blocksparse_attn_interface import convert_blockmask
    g = torch.Generator().manual_seed(0)
    for shape in ((1, 1), (3, 2), (7, 5), (16, 4), (256, 16)):
        for dens in (0.0, 0.2, 0.6, 1.0):
            m = torch.rand(shape, generator=g) < dens
            got = convert_blockmask(m, causal=False)
            assert got.dtype == torch.int32 and tuple(got.shape) == (shape[1], shape[0])
            assert np.array_equal(got.numpy(), orc.convert_blockmask_ref(m.numpy()))
    # causal (the reference asserts against it, flash_blocksparse_attn_interface.py:21): the list of the layout with
    # the blocks that hold no key <= query taken out, found here element by element
    for shape in ((3, 2), (16, 1), (40, 3), (64, 4)):
        m = torch.rand(shape, generator=g) < 0.7
        seen = np.zeros(shape, dtype=bool)
        for r in range(shape[0]):
            for c in range(shape[1]):
                seen[r, c] = any(k <= q for q in range(16 * r, 16 * r + 16) for k in (256 * c, 256 * c + 255))
        want = orc.convert_blockmask_ref(m.numpy() & seen)
        assert np.array_equal(convert_blockmask(m, causal=True).numpy(), want)


def test_unpad_pad_match_spec_and_backprop():
    from flash_attn.bert_padding import pad_input, unpad_input
    g = torch.Generator().manual_seed(1)
    x = torch.randn(3, 9, 6, generator=g, dtype=torch.float64, requires_grad=True)
    lens = torch.tensor([9, 4, 1])
    mask = torch.arange(9)[None, :] < lens[:, None]
    rows, idx, cu, mx = unpad_input(x, mask)
    r_rows, r_idx, r_cu, r_mx = orc.unpad_ref(x.detach().numpy(), mask.numpy())
    assert np.array_equal(rows.detach().numpy(), r_rows) and np.array_equal(idx.numpy(), r_idx)
    assert cu.dtype == torch.int32 and cu.tolist() == r_cu.tolist() and mx == r_mx
    back = pad_input(rows, idx, 3, 9)
    assert np.array_equal(back.detach().numpy(), orc.pad_ref(r_rows, r_idx, 3, 9))
    assert torch.equal(back.detach(), x.detach() * mask[..., None])  # pad(unpad(x)) == x o mask
    w = torch.randn(3, 9, 6, generator=g, dtype=torch.float64)
    (back * w).sum().backward()
    assert torch.equal(x.grad, w * mask[..., None])


def test_rotary_is_a_rotation_by_position_times_frequency():
    """closed form of rotary.py:22-42,66-87: pair i at position t is rotated by t * 10000^(-2i/dim)."""
    from flash_attn.rotary import RotaryEmbedding, RotaryEmbedding2D
    dim, S = 8, 5
    rot = RotaryEmbedding(dim)
    g = torch.Generator().manual_seed(2)
    q = torch.randn(2, 3, S, dim, generator=g, dtype=torch.float64)
    k = torch.randn(2, 3, S, dim, generator=g, dtype=torch.float64)
    rq, rk = rot(q, k)
    t = torch.arange(S, dtype=torch.float64)[:, None]
    ang = t * (10000.0 ** (-torch.arange(0, dim, 2, dtype=torch.float64) / dim))[None, :]
    zq = torch.view_as_complex(q.reshape(2, 3, S, dim // 2, 2).contiguous()) * torch.polar(torch.ones_like(ang), ang)
    assert torch.allclose(torch.view_as_real(zq).reshape(2, 3, S, dim), rq, atol=1e-6)
    # norms are preserved and q.k depends only on relative position
    assert torch.allclose(rq.norm(dim=-1), q.norm(dim=-1), atol=1e-6)
    q1 = torch.randn(dim, generator=g, dtype=torch.float64).expand(1, 1, S, dim).contiguous()
    k1 = torch.randn(dim, generator=g, dtype=torch.float64).expand(1, 1, S, dim).contiguous()
    a, b = RotaryEmbedding(dim)(q1, k1)
    dots = a[0, 0] @ b[0, 0].T
    assert torch.allclose(dots[1, 0], dots[3, 2], atol=1e-6) and torch.allclose(dots[0, 2], dots[2, 4], atol=1e-6)
    # layout (b, s, h, d) gives the same numbers as (b, h, s, d)
    rq2, _ = RotaryEmbedding(dim)(q.transpose(1, 2), k.transpose(1, 2), seq_dimension=-3)
    assert torch.allclose(rq2.transpose(1, 2), rq, atol=1e-12)
    # 2-D: first half of the channels rotates with the column index, second half with the row index
    side = 3
    x = torch.randn(1, 2, side * side, 8, generator=g, dtype=torch.float64)
    r2, _ = RotaryEmbedding2D(8)(x, x)
    one = RotaryEmbedding(4)
    grid = x.reshape(1, 2, side, side, 8)
    cols, _ = one(grid[..., :4], grid[..., :4], seq_dimension=-2)
    rows, _ = RotaryEmbedding(4)(grid[..., 4:].transpose(2, 3), grid[..., 4:].transpose(2, 3), seq_dimension=-2)
    want = torch.cat([cols, rows.transpose(2, 3)], dim=-1).reshape(1, 2, side * side, 8)
    assert torch.allclose(r2, want, atol=1e-12)


def test_blocksparse_module_layout_handling_on_host():
    """FlashBlocksparseAttention keeps the layout and its converted form as buffers (flash_blocksparse_attention.py:31-36)
    and accepts a tensor, a make_layout() object or, only with hydra installed, a _target_ mapping."""
    import importlib.util
    from flash_attn.flash_blocksparse_attention import FlashBlocksparseAttention
    layout = (torch.arange(48 * 3).reshape(48, 3) % 4 != 1).to(torch.int32)

    class Cfg:
        def make_layout(self, seqlen):
            assert seqlen == 768  # 700 rounded up to a multiple of 256
            return layout

    m = FlashBlocksparseAttention(Cfg(), max_seq_length=700)
    assert set(dict(m.named_buffers())) == {"layout", "blockmask_converted"}
    assert torch.equal(m.blockmask_converted, torch.tensor(orc.convert_blockmask_ref(layout.numpy())))
    assert tuple(m._blockmask(300).shape) == (19, 2) and tuple(m._blockmask(768).shape) == (48, 3)
    with pytest.raises(AssertionError):
        m._blockmask(769)
    with pytest.raises(ValueError):
        FlashBlocksparseAttention(layout[:10], max_seq_length=700)
    with pytest.raises(TypeError):
        FlashBlocksparseAttention("not a layout")
    if importlib.util.find_spec("hydra") is None:
        with pytest.raises(RuntimeError, match="hydra"):
            FlashBlocksparseAttention({"_target_": "some.module.Config"})


def test_dbias_layout_is_validated_before_anything_is_launched(lib):
    """every (batch, head) must have its own slice of dbias: overlapping slices would be written by several workgroups"""
    from flash_attn import flash_attn_gfx950 as be
    a = be.BwdArgs()
    a.struct_bytes = ctypes.sizeof(a)
    a.dtype = be.FA_FP16
    a.batch, a.nheads, a.head_dim = 2, 3, 64
    a.total_q = a.total_k = 64
    a.max_seqlen_q = a.max_seqlen_k = 32
    a.lse_seq_stride = 32
    a.p_dropout, a.softmax_scale = 0.0, 0.125
    fake = 0x10000  # never dereferenced: the checks below fail before any launch
    for f in ("dout", "q", "k", "v", "out", "softmax_lse", "dq", "dk", "dv", "softmax_d", "cu_seqlens_q", "cu_seqlens_k"):
        setattr(a, f, fake)
    for t in ("do", "q", "k", "v", "o", "dq", "dk", "dv"):
        setattr(a, t + "_row_stride", 192)
        setattr(a, t + "_head_stride", 64)
    a.attn_bias, a.bias_row_stride, a.bias_head_stride, a.bias_batch_stride = fake, 32, 32 * 32, 3 * 32 * 32
    a.dbias = fake
    good = dict(dbias_row_stride=32, dbias_head_stride=32 * 32, dbias_batch_stride=3 * 32 * 32)
    for field, value in (("dbias_row_stride", 24), ("dbias_head_stride", 31 * 32), ("dbias_head_stride", 0),
                         ("dbias_batch_stride", 2 * 32 * 32), ("dbias_batch_stride", 0)):
        for k, v in good.items():
            setattr(a, k, v)
        setattr(a, field, value)
        assert lib.fa_bwd(ctypes.byref(a)) == -1 and b"dbias needs its own slice" in lib.fa_last_error(), (field, value)
    for k, v in good.items():
        setattr(a, k, v)
    a.dbias = fake + 1
    assert lib.fa_bwd(ctypes.byref(a)) == -1 and b"2-byte alignment" in lib.fa_last_error()
    a.dbias, a.attn_bias = fake, None
    assert lib.fa_bwd(ctypes.byref(a)) == -1 and b"dbias without attn_bias" in lib.fa_last_error()


def test_in_kernel_rotary_arguments_are_validated_before_anything_is_launched(lib):
    """tables come in pairs, aligned, with a row for every position; not together with the probability dump"""
    from flash_attn import flash_attn_gfx950 as be
    fake = 0x10000  # never dereferenced: the checks below fail before any launch
    f = be.FwdArgs()
    f.struct_bytes = ctypes.sizeof(f)
    f.dtype = be.FA_FP16
    f.batch, f.nheads, f.head_dim = 2, 3, 64
    f.total_q = f.total_k = 64
    f.max_seqlen_q = f.max_seqlen_k = 32
    f.p_dropout, f.softmax_scale = 0.0, 0.125
    for name in ("q", "k", "v", "o", "softmax_lse", "cu_seqlens_q", "cu_seqlens_k"):
        setattr(f, name, fake)
    for t in ("q", "k", "v", "o"):
        setattr(f, t + "_row_stride", 192)
        setattr(f, t + "_head_stride", 64)
    f.rotary_cos, f.rotary_table_rows = fake, 32
    assert lib.fa_fwd(ctypes.byref(f)) == -1 and b"come together" in lib.fa_last_error()
    f.rotary_sin = fake + 8
    assert lib.fa_fwd(ctypes.byref(f)) == -1 and b"16-byte aligned" in lib.fa_last_error()
    f.rotary_sin, f.rotary_table_rows = fake, 31
    assert lib.fa_fwd(ctypes.byref(f)) == -1 and b"a row for every query position" in lib.fa_last_error()
    f.rotary_table_rows, f.s_dmask = 32, fake
    assert lib.fa_fwd(ctypes.byref(f)) == -4 and b"rotate with fa_rotary first" in lib.fa_last_error()
    f.s_dmask, f.q_rot, f.q_rot_row_stride, f.q_rot_head_stride = None, fake, 100, 64
    assert lib.fa_fwd(ctypes.byref(f)) == -1 and b"q_rot must be" in lib.fa_last_error()

    a = be.BwdArgs()
    a.struct_bytes = ctypes.sizeof(a)
    a.dtype = be.FA_FP16
    a.batch, a.nheads, a.head_dim = 2, 3, 64
    a.total_q = a.total_k = 64
    a.max_seqlen_q, a.max_seqlen_k = 32, 40
    a.lse_seq_stride = 32
    a.p_dropout, a.softmax_scale = 0.0, 0.125
    for name in ("dout", "q", "k", "v", "out", "softmax_lse", "dq", "dk", "dv", "softmax_d", "cu_seqlens_q", "cu_seqlens_k"):
        setattr(a, name, fake)
    for t in ("do", "q", "k", "v", "o", "dq", "dk", "dv"):
        setattr(a, t + "_row_stride", 192)
        setattr(a, t + "_head_stride", 64)
    a.rotary_sin, a.rotary_table_rows = fake, 40
    assert lib.fa_bwd(ctypes.byref(a)) == -1 and b"come together" in lib.fa_last_error()
    a.rotary_cos, a.rotary_table_rows = fake, 39
    assert lib.fa_bwd(ctypes.byref(a)) == -1 and b"a row for every query and key position" in lib.fa_last_error()


def test_launch_policy_values_and_one_kernel_backward_scratch(lib):
    """fa_set_launch_policy: tile shape in the low bits, backward plan in 0x30; the one-kernel backward asks for scratch only
    where it exists (head dim 64, dense, no mask, dropout or bias, at most 32 key tiles)"""
    from flash_attn import flash_attn_gfx950 as be
    for ok in (0, 1, 2, 0x10, 0x11, 0x12, 0x20, 0x21, 0x22, 0x40, 0x52):
        assert lib.fa_set_launch_policy(ok) == 0
    for bad in (3, 0x30, 0x80, 0x43, -1, 0x100):
        assert lib.fa_set_launch_policy(bad) == -1 and b"launch policy" in lib.fa_last_error()
    a = be.BwdArgs()
    a.struct_bytes = ctypes.sizeof(a)
    a.batch, a.nheads, a.head_dim = 8, 12, 64
    a.max_seqlen_q = a.max_seqlen_k = 2048
    try:
        lib.fa_set_launch_policy(0)
        assert lib.fa_bwd_workspace_bytes(ctypes.byref(a)) == 0      # the two-kernel backward needs no scratch
        lib.fa_set_launch_policy(0x20)
        want = 8 * 12 * 64 * (32 * 64 * 4 + 16)                      # fp32 running sums and four counters per 32-row tile
        assert lib.fa_bwd_workspace_bytes(ctypes.byref(a)) == want
        for field, value in (("head_dim", 128), ("is_causal", 1), ("p_dropout", 0.1), ("max_seqlen_k", 4097)):
            b = be.BwdArgs.from_buffer_copy(a)
            setattr(b, field, value)
            assert lib.fa_bwd_workspace_bytes(ctypes.byref(b)) == 0, field
    finally:
        lib.fa_set_launch_policy(0)


def test_key_split_workspace_plan(lib):
    """fa_fwd_workspace_bytes asks for scratch only for dense, non-causal forwards with one query tile and more keys than the
    (batch, head) pairs alone spread over the chip; the size is n_splits * (fp32 partial outputs + partial lse)."""
    from flash_attn import flash_attn_gfx950 as be
    a = _valid_fwd_args(be)
    a.batch, a.nheads, a.head_dim = 8, 12, 64
    a.total_q, a.total_k, a.max_seqlen_q, a.max_seqlen_k = 8, 8 * 2048, 1, 2048
    need = lib.fa_fwd_workspace_bytes(ctypes.byref(a))
    # 96 workgroups -> 8 splits of 4 key tiles; partial o: 8 x 8 x 12 x 64 fp32, partial lse: 8 x 8 x 12 x 16 fp32
    assert need == 8 * 8 * 12 * 64 * 4 + 8 * 8 * 12 * 16 * 4
    a.is_causal = 1
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) == 0
    a.is_causal = 0
    a.max_seqlen_q, a.total_q = 129, 8 * 129                   # more than one query tile per sequence
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) == 0
    a.max_seqlen_q, a.total_q, a.max_seqlen_k = 1, 8, 300      # too few keys to share
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) == 0
    a.max_seqlen_k, a.batch, a.total_q = 2048, 64, 64          # enough (batch, head) pairs to fill the chip
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) == 0
    # the backward asks for the fp32 partial dQ of the same plan (8 splits x 8 rows x 12 heads x 64), and for nothing
    # where the forward asks for nothing
    g = be.BwdArgs()
    g.struct_bytes = ctypes.sizeof(g)
    g.batch, g.nheads, g.head_dim = 8, 12, 64
    g.total_q, g.total_k, g.max_seqlen_q, g.max_seqlen_k = 8, 8 * 2048, 1, 2048
    assert lib.fa_bwd_workspace_bytes(ctypes.byref(g)) == 8 * 8 * 12 * 64 * 4
    g.is_causal = 1
    assert lib.fa_bwd_workspace_bytes(ctypes.byref(g)) == 0
    g.is_causal, g.max_seqlen_q, g.total_q = 0, 2048, 8 * 2048
    assert lib.fa_bwd_workspace_bytes(ctypes.byref(g)) == 0


@pytest.mark.parametrize("head_dim,batch,nheads,keys,mean,splits", [
    (128, 20, 16, 200, 1.0, 1), (128, 13, 16, 600, 1.0, 1), (16, 13, 16, 600, 1.0, 1),   # a merge would cost more than it saves
    (64, 1, 8, 512, 1.0, 1), (64, 1, 8, 513, 1.0, 3), (32, 1, 8, 1024, 1.0, 1), (32, 1, 8, 1025, 1.0, 3),  # eight rounds, nine
    (64, 16, 10, 600, 1.0, 4), (64, 16, 11, 600, 1.0, 1), (64, 16, 11, 1024, 1.0, 4),    # 160 pairs and more
    (128, 8, 12, 12000, 1.0, 5), (128, 8, 16, 12000, 1.0, 4), (128, 1, 8, 12000, 1.0, 32),  # whole workgroups per compute unit
    (128, 20, 16, 3000, 1.0, 1), (128, 20, 16, 3000, 0.6, 2), (64, 20, 16, 3000, 1.0, 2),   # uneven lengths leave room
    (128, 40, 16, 3000, 1.0, 1), (128, 64, 16, 3000, 1.0, 1), (64, 100, 16, 3000, 1.0, 1),  # the chip is full
])
def test_decode_split_plan(lib, head_dim, batch, nheads, keys, mean, splits):
    """The key splits of a decode step (one new token) by head dimension, pairs and keys, read off the scratch asked for."""
    from flash_attn import flash_attn_gfx950 as be
    a = _valid_fwd_args(be)
    a.batch, a.nheads, a.head_dim = batch, nheads, head_dim
    a.total_q, a.total_k, a.max_seqlen_q, a.max_seqlen_k = batch, int(batch * keys * mean), 1, keys
    per_split = batch * nheads * (head_dim + 16) * 4  # partial o, and partial lse with 16 rows
    assert lib.fa_fwd_workspace_bytes(ctypes.byref(a)) == (splits * per_split if splits > 1 else 0)


def test_rows_and_rotary_argument_checks(lib):
    """the byte-movement entry points reject bad arguments before any launch (CPU only: nothing valid is executed)"""
    from flash_attn import flash_attn_gfx950 as be
    assert lib.fa_scatter_rows_workspace_bytes(1000) == 4000 and lib.fa_scatter_rows_workspace_bytes(0) == 0
    assert lib.fa_gather_rows(0x1000, 0x2000, 0x3000, 4, 4, 64, 32, 64, None) == -1      # row stride < row width
    assert b"stride" in lib.fa_last_error()
    assert lib.fa_gather_rows(None, 0x2000, 0x3000, 4, 4, 64, 64, 64, None) == -1        # null source
    assert lib.fa_gather_rows(None, None, None, 0, 0, 64, 64, 64, None) == 0             # nothing to do
    assert lib.fa_scatter_rows(0x1000, 0x2000, 0x3000, 4, 8, 64, 64, 64, None, 0, None) == -2
    assert b"workspace" in lib.fa_last_error()
    assert lib.fa_scatter_rows(0x1000, 0x2000, 0x3000, 4, -1, 64, 64, 64, 0x4000, 64, None) == -1
    r = be.RotaryArgs()
    r.struct_bytes = ctypes.sizeof(r) - 4
    assert lib.fa_rotary(ctypes.byref(r)) == -1 and b"struct size" in lib.fa_last_error()
    r.struct_bytes = ctypes.sizeof(r)
    r.dtype, r.n_rows, r.n_parts, r.n_rotated, r.n_heads, r.head_dim = 0, 4, 3, 2, 2, 12
    assert lib.fa_rotary(ctypes.byref(r)) == -1 and b"multiple of 8" in lib.fa_last_error()
    r.head_dim, r.n_rotated = 64, 4
    assert lib.fa_rotary(ctypes.byref(r)) == -1 and b"sizes" in lib.fa_last_error()
    r.n_rotated = 2
    assert lib.fa_rotary(ctypes.byref(r)) == -1 and b"null" in lib.fa_last_error()
    r.n_rows = 0
    assert lib.fa_rotary(ctypes.byref(r)) == 0
    assert lib.fa_token_positions(0x1000, 0, 4, 0x2000, None) == -1 and b"sizes" in lib.fa_last_error()
    assert lib.fa_token_positions(None, 1, 4, 0x2000, None) == -1 and b"null" in lib.fa_last_error()
    assert lib.fa_token_positions(0x1000, 1, 4, 0x2002, None) == -1 and b"aligned" in lib.fa_last_error()
    assert lib.fa_token_positions(None, 1, 0, None, None) == 0


def test_bias_grad_reduce_argument_checks(lib):
    """fa_bias_grad_reduce rejects bad arguments before any launch (CPU only: nothing valid is executed)"""
    ok_in = (2, 3, 16, 20, 3 * 16 * 24, 16 * 24, 24)   # batch, heads, rows, cols, dbias strides (rows padded to 24 columns)
    ok_out = (1, 0, 3 * 16 * 20, 16 * 20, 20)          # sum_batch, sum_heads, out strides
    call = lambda dbias, out, dtype, i, o: lib.fa_bias_grad_reduce(dbias, out, dtype, *i, *o, None)
    assert call(0x1000, 0x2000, 2, ok_in, ok_out) == -1 and b"dtype" in lib.fa_last_error()
    assert call(None, 0x2000, 0, ok_in, ok_out) == -1 and b"null" in lib.fa_last_error()
    assert call(0x1008, 0x2000, 0, ok_in, ok_out) == -1 and b"aligned" in lib.fa_last_error()            # 8-byte aligned only
    assert call(0x1000, 0x2000, 0, (2, 3, 16, 20, 3 * 16 * 20, 16 * 20, 20), ok_out) == -1               # rows not padded to 8
    assert call(0x1000, 0x2000, 0, ok_in, (1, 0, 3 * 16 * 20, 16 * 20, 19)) == -1 and b"out row" in lib.fa_last_error()
    assert call(0x1000, 0x2000, 0, (70000, 3, 16, 20, 3 * 16 * 24, 16 * 24, 24), ok_out) == -1
    assert call(None, None, 1, (0, 3, 16, 20, 0, 0, 24), ok_out) == 0                                    # nothing to do
    assert call(None, None, 1, (2, 3, 16, 0, 0, 0, 0), ok_out) == 0


def test_bias_rows_launch_fits_a_grid_at_every_size(tmp_path):
    """The launch that pads a bias tensor's rows stays below the 2^32 threads a grid may hold and covers every group of rows once, up to
    tensors of billions of rows (host code of the library's own header; nothing is launched)."""
    import subprocess
    import build as fa_build
    src, exe = tmp_path / "grid.hip", tmp_path / "grid"
    src.write_text("""#include <cstdio>
#include "fa_params.h"
int main() {
  const int64_t sizes[][3] = {{1, 1, 1}, {1, 12, 333}, {8, 16, 1101}, {64, 16, 65535}, {64, 16, 65536}, {128, 16, 65537}, {1, 1, 3000000000}};
  for (auto& s : sizes) {
    const fa::PadBiasGrid g = fa::pad_bias_grid((int)s[0], (int)s[1], s[2]);
    std::printf("%lld %lld %lld %lld %lld %u\\n", (long long)s[0], (long long)s[1], (long long)s[2], (long long)g.row_groups, (long long)g.groups, g.blocks);
  }
}
""".replace("\\\\n", "\\n"))
    cmd = [fa_build.HIPCC, "--offload-host-only", "-std=c++17", "-I", fa_build.CSRC, str(src), "-o", str(exe)]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    lines = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, check=True).stdout.splitlines()
    assert len(lines) == 7
    for line in lines:
        nb, nh, rows, row_groups, groups, blocks = map(int, line.split())
        assert row_groups == -(-rows // 4) and groups == nb * nh * row_groups
        assert 0 < blocks <= groups and blocks * 256 < 1 << 32
        assert blocks == groups or blocks >= 1 << 20  # (one workgroup a group, as measured, unless there are more than a grid holds)


def test_pad_bias_rows_argument_checks(lib):
    """fa_pad_bias_rows: what it refuses, and that large tensors are not among it (a null pointer is what these are refused for)"""
    call = lambda *sizes: lib.fa_pad_bias_rows(None, None, *sizes, 1, 1, 1, 1, None)
    assert call(0, 3, 4, 5) == 0 and call(2, 3, 0, 5) == 0
    for sizes in ((-1, 1, 1, 1), (1, 1, -1, 1), (1, 1, 1, 1 << 32), (1 << 30, 1 << 30, 9, 1)):
        assert call(*sizes) == -1 and b"null" not in lib.fa_last_error(), sizes
    for sizes in ((64, 16, 65536, 77), (64, 64, 1 << 20, 8), (1, 1, 1 << 31, 8), (1, 1, 1, 1 << 30)):
        assert call(*sizes) == -1 and b"null" in lib.fa_last_error(), sizes


def test_header_is_plain_c(tmp_path):
    """include/flash_attn_gfx950.h must be usable from C (the boundary a cgo / JNI / ctypes binding sees): it compiles as
    C99 with warnings as errors, and every declared entry point can be named."""
    import subprocess
    from flash_attn import flash_attn_gfx950 as be
    src = tmp_path / "use_header.c"
    names = [n for n in be.EXPORTED_SYMBOLS]
    src.write_text('#include "flash_attn_gfx950.h"\n'
                   "typedef void (*entry_t)(void);\n"
                   "entry_t entry_points[] = {" + ", ".join("(entry_t)%s" % n for n in names) + "};\n"
                   "int sizes[] = {(int)sizeof(fa_fwd_args), (int)sizeof(fa_bwd_args), (int)sizeof(fa_rotary_args)};\n")
    r = subprocess.run(["gcc", "-std=c99", "-Wall", "-Wextra", "-Werror", "-pedantic", "-fsyntax-only",
                        "-I", os.path.join(ROOT, "include"), str(src)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout



def test_prepare_attn_bias_layout_rules():
    """prepare_attn_bias hands the caller's tensor through when the kernels can read it as it is (keys contiguous, rows a
    multiple of 8 elements, 16-byte aligned) and pads a copy otherwise; shape, dtype and device are checked."""
    from flash_attn import flash_attn_gfx950 as be
    q = torch.zeros(10, 3, 64, dtype=torch.float16)
    good = torch.randn(1, 3, 40, 48).half()
    assert be.prepare_attn_bias(good, q, 2, 3, 40, 48) is good
    assert be.prepare_attn_bias(good, q, 2, 3, 33, 41) is good                       # larger than needed is fine
    odd = torch.randn(2, 1, 40, 45).half()
    p = be.prepare_attn_bias(odd, q, 2, 3, 40, 45)
    assert p is not odd and tuple(p.shape) == (2, 1, 40, 48) and p.stride(2) % 8 == 0 and p.stride(3) == 1
    assert torch.equal(p[..., :45], odd) and torch.equal(p[..., 45:], torch.zeros(2, 1, 40, 3).half())
    view = torch.randn(1, 3, 40, 96).half()[..., ::2]                                  # keys not contiguous
    p = be.prepare_attn_bias(view, q, 2, 3, 40, 48)
    assert p.stride(3) == 1 and torch.equal(p, view)
    for bad, msg in ((torch.zeros(3, 3, 40, 48).half(), "attn_bias must be"),           # batch neither 1 nor 2
                     (torch.zeros(1, 2, 40, 48).half(), "attn_bias must be"),           # heads neither 1 nor 3
                     (torch.zeros(1, 3, 39, 48).half(), "attn_bias must be"),           # too few rows
                     (torch.zeros(1, 3, 40, 47).half(), "attn_bias must be"),           # too few keys
                     (torch.zeros(3, 40, 48).half(), "attn_bias must be"),              # not 4-D
                     (torch.zeros(1, 3, 40, 48), "dtype and device")):                  # fp32 for fp16 inputs
        with pytest.raises(RuntimeError, match=msg):
            be.prepare_attn_bias(bad, q, 2, 3, 40, 48)


def test_drawn_philox_state_survives_as_a_saved_tensor():
    from flash_attn.flash_attn_gfx950 import DrawnPhilox
    for state in ((0, 0), (5, 4), (1 << 63, 8), ((1 << 64) - 1, (1 << 63) + 12)):
        d = DrawnPhilox()
        d.state = state
        t = d.saved()
        assert t.device.type == "cpu" and t.dtype == torch.int64 and DrawnPhilox(t.clone()).state == state


def test_dropout_state_is_saved_as_tensors_where_hooks_see_them(monkeypatch):
    from flash_attn import flash_attn_gfx950 as be
    d, words = be.DrawnPhilox(), torch.zeros(4, dtype=torch.uint8)
    d.state = (7, 8)
    saved, kept = be.pack_dropout(words, d)
    assert be.unpack_dropout(saved, kept) == (words, d)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert be.pack_dropout(None, None) == ((None, None), (None, None))  # (no dropout: nothing to save)
        saved, kept = be.pack_dropout(words, d)
    assert kept is None and saved[0] is words
    got = be.unpack_dropout(saved, kept)
    assert got[0] is words and got[1].state == (7, 8)
    monkeypatch.setattr(be, "_saved_tensor_hooks", None)
    assert be.pack_dropout(words, d)[1] is None


def _launch_rules(tmp_path, expressions):
    """Values of expressions over the launch rules of fa_params.h under the default policy (host code; nothing is launched)"""
    import subprocess
    import build as fa_build
    src, exe = tmp_path / "rules.hip", tmp_path / "rules"
    src.write_text('#include <cstdio>\n#include "fa_params.h"\nnamespace fa { int launch_policy() { return 0; } }\nusing namespace fa;\n'
                   'int main() {\n' + "".join('  std::printf("%%d\\n", (int)(%s));\n' % e for e in expressions) + "}\n")
    cmd = [fa_build.HIPCC, "--offload-host-only", "-std=c++17", "-I", fa_build.CSRC, str(src), "-o", str(exe)]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    return [int(x) for x in subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, check=True).stdout.split()]


def _spread(n, frac, batch):
    """tokens of a batch whose lengths are spread evenly between frac * n and n"""
    return sum(int(n - (n - frac * n) * i // max(1, batch - 1)) for i in range(batch))


def test_d128_forward_tiles_follow_the_measurements(tmp_path):
    """head dim 128: full- or half-size tiles by what was faster, us full / half, where the difference is more than the measurement's noise"""
    cases = [  # batch, heads, longest, shortest / longest, causal, half-size?
        (8, 16, 281, 1.0, 1, 0), (16, 8, 286, 1.0, 1, 0), (12, 12, 305, 0.55, 1, 0), (10, 12, 337, 0.77, 1, 0), (10, 12, 287, 0.66, 1, 0),  # 12.8 / 15.7 ..
        (8, 12, 386, 0.86, 1, 0), (12, 8, 409, 1.0, 1, 0), (16, 8, 158, 0.53, 1, 0),  # 15.7 / 17.0, 16.0 / 18.0, 8.2 / 8.7
        (6, 8, 323, 1.0, 0, 0), (3, 16, 325, 1.0, 0, 0), (4, 8, 531, 1.0, 0, 0),  # 12.4 / 13.9, 12.0 / 13.4, 16.1 / 17.1
        (1, 8, 2300, 1.0, 1, 1), (4, 12, 1200, 0.3, 1, 1), (4, 16, 300, 1.0, 1, 1), (1, 16, 3000, 1.0, 1, 1),  # 53.9 / 35.8, 32.7 / 24.8, 11.9 / 11.0, 69.8 / 51.4
        (1, 8, 1700, 1.0, 0, 1), (3, 16, 286, 1.0, 0, 1)]  # 39.3 / 28.1, 10.8 / 10.0
    rotary = [(12, 8, 197, 0.75, 1, 0), (6, 16, 276, 1.0, 1, 0), (9, 8, 229, 0.43, 0, 0), (3, 8, 706, 0.91, 0, 0),  # 12.0 / 14.4 .. 23.1 / 24.7
              (1, 8, 2300, 1.0, 1, 1), (1, 8, 1100, 1.0, 0, 1), (2, 8, 500, 1.0, 1, 1)]
    for rot, cs in ((0, cases), (1, rotary)):
        got = _launch_rules(tmp_path, ["small_launch_d128(live_row_tiles(%d, %d, %d), %d, %d, %d, %d, %d)" % (h, _spread(n, f, b), b, b * h, n, n, c, rot)
                                       for b, h, n, f, c, _ in cs])
        assert got == [c[-1] for c in cs], [c for c, g in zip(cs, got) if g != c[-1]]
    # fewer keys than queries: us full / half 20.3 / 26.0, 27.9 / 31.1, 7.5 / 8.0; as many or more keys as above
    got = _launch_rules(tmp_path, ["small_launch_d128(live_row_tiles(%d, %d, %d), %d, %d, %d, %d, 0)" % (h, b * n, b, b * h, n, k, c) for b, h, n, k, c in (
        (1, 12, 2413, 603, 1), (3, 8, 1736, 868, 1), (2, 16, 352, 88, 0), (1, 8, 2300, 4600, 1), (1, 8, 1700, 1700, 0))])
    assert got == [0, 0, 0, 1, 1]


def _rule_case(b, h, n, f):
    return "live_row_tiles(%d, %d, %d), %d, %d, %d" % (h, _spread(n, f, b), b, b * h, n, n)


def test_d64_backward_in_one_launch_where_measured(tmp_path):
    """head dim 64: dQ and dK/dV in one launch or two by what was faster, us in two (full-size) / in one; where dropout is read from keep words, two
    launches run the full-size tiles"""
    cases = [  # batch, heads, longest, shortest / longest, causal, dropout, one launch?
        (1, 16, 3616, 1.0, 0, 0, 0), (1, 8, 7464, 1.0, 0, 0, 0), (1, 12, 3768, 1.0, 0, 0, 0), (3, 16, 1203, 1.0, 0, 0, 0),  # 195 / 219 .. 77 / 84
        (7, 16, 239, 1.0, 0, 0, 0), (5, 16, 277, 1.0, 0, 0, 0), (5, 16, 667, 1.0, 0, 0, 0), (8, 16, 392, 1.0, 0, 0, 0),  # 20.4 / 21.6 .. 36.7 / 38.5
        (27, 8, 273, 1.0, 1, 0, 0), (15, 8, 585, 1.0, 1, 0, 0), (16, 16, 219, 1.0, 1, 0, 0), (16, 8, 602, 1.0, 1, 1, 0),  # 30.5 / 33.4 .. 48.1 / 51.1
        (4, 8, 2013, 1.0, 0, 1, 0), (21, 12, 81, 0.905, 0, 1, 0), (32, 16, 76, 1.0, 1, 0, 0), (16, 12, 70, 1.0, 0, 0, 0),  # 142 / 150, 17.2 / 19.0
        (33, 12, 73, 1.0, 0, 1, 1), (17, 16, 123, 1.0, 0, 1, 1), (36, 12, 108, 1.0, 0, 1, 1), (27, 16, 110, 1.0, 1, 1, 1),  # 23.5 / 22.1, 22.8 / 19.4
        (33, 12, 115, 1.0, 1, 0, 1), (16, 12, 97, 1.0, 1, 0, 1), (12, 16, 45, 1.0, 0, 0, 1),  # 22.7 / 21.3, 16.4 / 10.6, 12.7 / 9.3
        (1, 12, 1812, 1.0, 1, 0, 1), (4, 8, 2383, 1.0, 1, 0, 1), (3, 8, 846, 1.0, 0, 0, 1), (3, 16, 641, 1.0, 0, 0, 1),  # 75 / 50, 136 / 124, 40 / 26
        (11, 8, 276, 1.0, 0, 0, 1), (7, 16, 711, 0.535, 0, 1, 1), (8, 12, 731, 0.54, 0, 0, 1), (2, 8, 3441, 0.34, 0, 0, 1)]  # 29.0 / 23.1, 64.6 / 59.8
    one = _launch_rules(tmp_path, ["merged_backward_shape(64, %s, %d, %d, %d, 0, 0, 0, 1)" % (_rule_case(*c[:4]), c[4], c[5], c[5]) for c in cases])
    assert one == [c[-1] for c in cases], [c for c, g in zip(cases, one) if g != c[-1]]
    words = [c for c in cases if c[5]]
    half = _launch_rules(tmp_path, ["small_launch_dq(64, %s, %d, 1, 1, 0, 1)" % (_rule_case(*c[:4]), c[4]) for c in words])
    assert half == [c[-1] for c in words], [c for c, g in zip(words, half) if g != c[-1]]


def test_dq_tiles_follow_the_measurements(tmp_path):
    """dQ in a launch of its own, no dropout: full- or half-size tiles by what was faster, us of the backward full / half"""
    cases = [  # head dim, batch, heads, longest, shortest / longest, causal, half-size?
        (32, 17, 16, 115, 1.0, 1, 1), (32, 30, 12, 118, 1.0, 1, 1), (16, 22, 16, 74, 1.0, 1, 1), (16, 2, 8, 3964, 1.0, 1, 1),  # 15.8 / 15.1, 96.9 / 89.0
        (128, 7, 12, 135, 1.0, 0, 0), (128, 9, 8, 244, 0.33, 0, 0), (128, 6, 16, 509, 1.0, 1, 0), (32, 12, 16, 60, 1.0, 0, 0),  # 25.3 / 27.8, 29.6 / 30.3
        (128, 2, 8, 928, 1.0, 0, 1), (128, 1, 8, 974, 1.0, 1, 1), (128, 2, 12, 1500, 1.0, 1, 1), (32, 2, 16, 707, 0.46, 1, 1)]  # 67.6 / 60.5, 73.4 / 64.2
    half = _launch_rules(tmp_path, ["small_launch_dq(%d, %s, %d, 0, 0, 0, 1)" % (c[0], _rule_case(*c[1:5]), c[5]) for c in cases])
    assert half == [c[-1] for c in cases], [c for c, g in zip(cases, half) if g != c[-1]]
    assert _launch_rules(tmp_path, ["small_launch_dq(128, live_row_tiles(16, 2218, 2), 32, 1109, %d, 1, 0, 0, 0, 1)" % k for k in (277, 1109)]) == [0, 1]
    rotary = [(6, 8, 1012, 1.0, 1, 1), (3, 8, 2177, 1.0, 1, 1), (1, 16, 3394, 1.0, 1, 1), (18, 16, 126, 1.0, 1, 1),  # 57.6 / 53.1 .. 26.3 / 25.4
              (27, 16, 90, 1.0, 1, 0), (12, 8, 609, 1.0, 1, 0), (8, 12, 460, 1.0, 1, 1)]
    half = _launch_rules(tmp_path, ["small_launch_dq(64, %s, %d, 0, 0, 1, 1)" % (_rule_case(*c[:4]), c[4]) for c in rotary])
    assert half == [c[-1] for c in rotary], [c for c, g in zip(rotary, half) if g != c[-1]]


def test_causal_forward_tiles_follow_the_measurements(tmp_path):
    """head dim 16 to 64, causal: full- or half-size tiles by what was faster, us full / half"""
    cases = [  # head dim, batch, heads, longest, shortest / longest, half-size?
        (64, 16, 12, 329, 1.0, 0), (64, 11, 16, 355, 1.0, 0), (64, 8, 16, 527, 1.0, 0), (64, 7, 12, 838, 1.0, 0),  # 11.7 / 12.9 .. 19.7 / 21.1
        (64, 21, 12, 290, 0.64, 0), (64, 13, 16, 266, 1.0, 0), (64, 4, 12, 2300, 1.0, 0), (64, 4, 12, 1700, 1.0, 0),  # 11.4 / 12.9, 10.9 / 11.9
        (64, 20, 8, 364, 1.0, 1), (64, 3, 12, 1823, 1.0, 1), (64, 3, 12, 2829, 0.49, 1), (64, 6, 12, 1631, 0.16, 1),  # 11.2 / 10.5, 33.6 / 29.5
        (64, 16, 8, 1200, 0.4, 1), (32, 24, 8, 330, 0.9, 1), (16, 21, 8, 317, 1.0, 1)]  # 34.9 / 26.8, 9.3 / 9.0, 8.5 / 7.4
    half = _launch_rules(tmp_path, ["small_launch_causal(%d, live_row_tiles(%d, %d, %d), %d, %d, %d, %d)" % (
        d, h, _spread(n, f, b), b, b * h, n, _spread(n, f, b), b) for d, b, h, n, f, _ in cases])
    assert half == [c[-1] for c in cases], [c for c, g in zip(cases, half) if g != c[-1]]


def test_native_calls_leave_no_exception_behind_what_they_hand_back():
    """numbers a double cannot hold and flags without a truth value are handed back to the binding, which raises for them"""
    import numpy as np
    from flash_attn import flash_attn_gfx950 as be
    be.load_library()
    x, cu = torch.zeros(4, 2, 16, dtype=torch.half), torch.tensor([0, 4], dtype=torch.int32)
    for p, scale, zero, causal in ((10 ** 400, 0.1, False, False), (0.0, 10 ** 400, False, False), (0.0, 0.1, np.ones(2), False),
                                   (0.0, 0.1, False, np.ones(2))):
        assert be._host.fwd(x, x, x, cu, cu, 4, 4, p, scale, zero, causal, *[None] * 9) is None
        assert be._host.bwd(x, x, x, x, x, None, x, x, x, cu, cu, 4, 4, p, scale, zero, causal, *[None] * 9) is None


def test_padded_forward_tiles_follow_the_measurements(tmp_path):
    """padded batches: full- or half-size tiles by what was faster over batches of 30 % to 100 % tokens"""
    cases = [  # head dim, batch, heads, rows, causal, half-size?
        (128, 6, 16, 400, 1, 1), (128, 4, 12, 1079, 1, 1), (128, 2, 12, 1217, 1, 1), (128, 1, 16, 1376, 0, 1),  # us full / half: 16.1 / 14.4 .. 36.2 / 31.2
        (128, 8, 12, 156, 0, 0), (128, 12, 16, 209, 0, 0), (128, 8, 16, 272, 1, 0), (128, 16, 8, 1500, 1, 0), (64, 32, 16, 512, 0, 0), (64, 8, 8, 512, 0, 1)]  # 10.3 / 11.7, 13.5 / 15.6
    half = _launch_rules(tmp_path, ["small_launch_rows(%d, %d, %d, %d, %d)" % c[:-1] for c in cases])
    assert half == [c[-1] for c in cases], [c for c, g in zip(cases, half) if g != c[-1]]


def test_live_order_not_where_it_reads_keys_again(tmp_path):
    """ragged causal launches of many pairs, whose K and V the groups of the other order keep in L2: us in groups / live"""
    cases = [  # kernel, head dim, batch, heads, longest, shortest / longest, live order?
        ("kLiveFwd", 128, 64, 16, 1024, 0.6, 0), ("kLiveFwd", 128, 64, 16, 2048, 0.3, 0), ("kLiveFwd", 128, 32, 16, 2048, 0.6, 0),  # 286 / 409, 675 / 953, 459 / 541
        ("kLiveFwd", 64, 64, 16, 2048, 0.6, 0), ("kLiveFwd", 64, 63, 8, 2463, 0.8, 0), ("kLiveFwd", 32, 20, 12, 4096, 0.6, 0),  # 509 / 640, 383 / 444, 281 / 366
        ("kLiveFwd", 16, 20, 12, 7900, 0.6, 0), ("kLiveDq", 16, 20, 12, 7900, 0.6, 0), ("kLiveDq", 32, 20, 12, 4096, 0.6, 0),  # 1009 / 1216, 1026 / 1314, 331 / 396
        ("kLiveDq", 64, 64, 16, 2048, 0.6, 0), ("kLiveDq", 128, 64, 16, 2048, 0.3, 0), ("kLiveDq", 128, 41, 16, 2261, 0.73, 0),  # 699 / 822, 992 / 1254, 1142 / 1443
        ("kLiveDkdv", 64, 31, 16, 3723, 0.65, 0), ("kLiveDkdv", 64, 36, 16, 3719, 0.48, 0),  # 1324 / 1440, 1299 / 1407
        ("kLiveFwd", 64, 32, 16, 2048, 0.3, 1), ("kLiveFwd", 128, 16, 8, 4096, 0.3, 1), ("kLiveFwd", 32, 7, 12, 7900, 0.3, 1),  # 215 / 192, 366 / 271, 279 / 246
        ("kLiveDq", 128, 64, 12, 520, 0.8, 1), ("kLiveDq", 64, 32, 16, 2048, 0.3, 1), ("kLiveDkdv", 128, 64, 8, 1024, 0.3, 1),  # 185 / 159, 292 / 239, 235 / 191
        ("kLiveDkdv", 64, 64, 16, 1024, 0.3, 1), ("kLiveDkdv", 128, 20, 12, 4096, 0.3, 1)]  # 219 / 195, 1327 / 1061

    def group(d, b, h, n):  # causal_tile_group
        kv, pairs = 4 * n * d, -(-b * h // 8)
        return 0 if pairs * kv <= 8 << 20 else max(4, (6 << 20) // kv)

    got = _launch_rules(tmp_path, ["live_order_launch(%s, %d, 1, %d, %d, %d, %d, 1, %d, %d, %d)" % (
        k, d, b, h, _spread(n, f, b), n, -(-n // 128), group(d, b, h, n), -(-b * h // 8) * 8 * -(-n // 128)) for k, d, b, h, n, f, _ in cases])
    assert got == [c[-1] for c in cases], [c for c, g in zip(cases, got) if g != c[-1]]


def test_live_order_where_measured(tmp_path):
    """ragged launches whose workgroups enumerate the tiles that hold rows, and those that keep the slot orders"""
    cases = [  # kernel, head dim, causal, batch, heads, longest, shortest / longest, tile_group, grid, live order?
        ("kLiveFwd", 128, 1, 4, 16, 3001, 0.2, 4, 1536, 1), ("kLiveFwd", 64, 0, 12, 12, 550, 0.39, 0, 720, 1), ("kLiveDq", 64, 1, 4, 12, 6000, 0.3, 4, 2256, 1),
        ("kLiveDkdv", 64, 1, 3, 16, 5841, 0.483, 4, 2208, 1), ("kLiveMerged", 64, 0, 8, 12, 512, 0.5, 0, 1152, 1), ("kLiveDkdv", 64, 0, 57, 8, 139, 0.39, 0, 912, 1),
        ("kLiveFwd", 64, 0, 64, 16, 1023, 0.982, 0, 8192, 0), ("kLiveFwd", 64, 0, 65, 8, 500, 0.5, 0, 2080, 0), ("kLiveFwd", 64, 0, 2, 8, 8193, 0.5, 0, 1040, 0),
        ("kLiveMerged", 64, 0, 3, 12, 910, 0.455, 0, 960, 0), ("kLiveMerged", 64, 1, 8, 12, 512, 0.5, 0, 1152, 0), ("kLiveFwd", 64, 1, 38, 16, 628, 0.66, 0, 3040, 0),
        ("kLiveFwd", 64, 1, 64, 8, 109, 0.383, 0, 512, 0), ("kLiveFwd", 64, 1, 2, 12, 787, 0.703, 0, 168, 0), ("kLiveDkdv", 64, 1, 14, 16, 703, 0.67, 0, 1344, 0),
        ("kLiveFwd", 32, 1, 64, 16, 926, 0.55, 53, 8192, 0)]
    got = _launch_rules(tmp_path, ["live_order_launch(%s, %d, %d, %d, %d, %d, %d, 1, %d, %d, %d)" % (
        k, d, c, b, h, _spread(n, f, b), n, -(-n // 128), group, grid) for k, d, c, b, h, n, f, group, grid, _ in cases])
    assert got == [c[-1] for c in cases], [c for c, g in zip(cases, got) if g != c[-1]]
    assert _launch_rules(tmp_path, ["live_order_launch(kLiveFwd, 64, 0, 4, 8, 1000, 1000, 2, 8, 0, 256)", "live_order_rows(64, 64)", "live_order_rows(65, 1)",
                                    "live_order_rows(1, 65)"]) == [0, 1, 0, 0]


def test_live_order_not_where_launches_are_short(tmp_path):
    """ragged causal launches without groups: of few workgroups, of half-size tiles just over a round of the chip, of fuller slots at head dim 128"""
    cases = [  # kernel, head dim, batch, heads, longest, shortest / longest, rows of a tile, live order?
        ("kLiveFwd", 64, 4, 12, 400, 0.86, 64, 0), ("kLiveFwd", 16, 12, 3, 1147, 0.55, 64, 0), ("kLiveFwd", 16, 12, 5, 557, 0.26, 64, 0),  # us in the slot order / live:
        ("kLiveFwd", 32, 6, 5, 1056, 0.71, 64, 0), ("kLiveFwd", 32, 8, 12, 464, 0.39, 64, 0), ("kLiveDq", 32, 2, 12, 2671, 0.51, 64, 0),  # 8.1 / 8.5, 10.7 / 11.2, 7.2 / 7.7,
        ("kLiveDq", 128, 12, 3, 593, 0.65, 64, 0), ("kLiveFwd", 64, 12, 12, 928, 0.22, 64, 0), ("kLiveFwd", 64, 3, 24, 1864, 0.31, 64, 0),  # 10.6 / 11.3, 7.5 / 7.9, 69.5 / 73.5,
        ("kLiveFwd", 128, 4, 8, 2384, 0.77, 128, 0), ("kLiveFwd", 128, 8, 8, 1195, 0.78, 128, 0), ("kLiveDq", 128, 8, 5, 920, 0.84, 64, 0),  # 48.3 / 49.4, 18.9 / 20.6, 28.8 / 31.2, ..
        ("kLiveFwd", 64, 2, 24, 3139, 0.15, 64, 1), ("kLiveFwd", 64, 5, 12, 3299, 0.3, 128, 1), ("kLiveFwd", 128, 12, 5, 1209, 0.2, 64, 1),  # 51.5 / 45.5, 81.0 / 61.0, 32.2 / 24.6
        ("kLiveFwd", 32, 12, 5, 1738, 0.2, 64, 1), ("kLiveFwd", 64, 6, 5, 3653, 0.17, 64, 1), ("kLiveDq", 32, 12, 12, 1230, 0.4, 64, 1)]
    got = _launch_rules(tmp_path, ["live_order_launch(%s, %d, 1, %d, %d, %d, %d, 1, %d, 0, %d)" % (
        k, d, b, h, _spread(n, f, b), n, -(-n // rows), -(-b * h // 8) * 8 * -(-n // rows)) for k, d, b, h, n, f, rows, _ in cases])
    assert got == [c[-1] for c in cases], [c for c, g in zip(cases, got) if g != c[-1]]


def test_live_order_batches_of_the_gpu_tests_take_it(tmp_path):
    """forward, dQ and dK/dV of the batch on which the variants are compared (16 heads, 1500 tokens and 31 sequences of 300 to 510), in full-size and
    half-size tiles, with a causal mask and without; not with 33 empty sequences behind it"""
    lens = [1500] + [300 + 7 * i for i in range(31)]
    n, total, expressions = max(lens), sum(lens), []
    for d in (64, 128):
        group = max(4, (6 << 20) // (4 * n * d))  # causal_tile_group: 64 pairs of an XCD are beyond its L2
        for causal in (0, 1):
            for rows in (128, 64):
                tiles = -(-n // rows)
                for kernel in ("kLiveFwd", "kLiveDq") + (("kLiveDkdv",) if rows == 128 else ()):
                    expressions += ["live_order_launch(%s, %d, %d, %d, 16, %d, %d, 1, %d, %d, %d)" % (
                        kernel, d, causal, b, total, n, tiles, group * causal, b * 16 * tiles) for b in (32, 65)]
    assert _launch_rules(tmp_path, expressions) == [1, 0] * (len(expressions) // 2)


def test_live_order_of_padded_batches_where_measured(tmp_path):
    """the forward over a padded batch: us in the slot order (groups) / live, all rows tokens or 30 % of them and more"""
    cases = [  # head dim, causal, batch, heads, rows, live order?
        (64, 1, 64, 16, 2048, 0), (64, 1, 32, 24, 2197, 0), (32, 1, 36, 16, 3218, 0), (32, 1, 33, 8, 4321, 0),  # 728 / 1028, 654 / 839, 718 / 983, 543 / 661
        (32, 1, 21, 16, 3933, 0), (16, 1, 7, 24, 7411, 0), (16, 1, 44, 8, 5687, 0), (16, 1, 40, 16, 533, 0),  # 590 / 785, 858 / 1131, 1129 / 1459, 42.9 / 45.8
        (64, 1, 16, 3, 172, 0), (64, 1, 14, 12, 300, 0), (16, 1, 28, 8, 183, 0), (64, 1, 4, 3, 162, 0),  # 6.4 / 7.0, 9.8 / 10.2, 5.9 / 6.3, 6.2 / 6.5
        (64, 0, 1, 5, 1865, 0), (32, 0, 1, 8, 795, 0), (64, 1, 65, 16, 512, 0), (64, 0, 65, 16, 512, 0),  # 21.1 / 21.7, 9.6 / 9.8
        (64, 1, 8, 12, 2048, 1), (64, 1, 16, 16, 4096, 1), (64, 1, 30, 12, 786, 1),  # 70.3 / 67.8, 688 / 674, 62.0 / 54.5
        (16, 1, 4, 8, 4720, 1), (64, 0, 64, 16, 512, 1), (64, 0, 46, 3, 197, 1), (32, 0, 62, 8, 2120, 1)]  # 70.1 / 51.9, 75.6 / 68.5, ..
    got = _launch_rules(tmp_path, ["live_order_padded(%d, %d, %d, %d, %d, %d)" % (d, c, b, h, n, -(-n // 128)) for d, c, b, h, n, _ in cases])
    assert got == [c[-1] for c in cases], [c for c, g in zip(cases, got) if g != c[-1]]
    # the GPU test of the order, whose causal batches are to take it
    assert _launch_rules(tmp_path, ["live_order_padded(32, 1, 12, 8, 700, 11)", "live_order_padded(64, 1, 9, 16, 600, 10)"]) == [1, 1]
