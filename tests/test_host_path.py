"""The operators' C++ host path without a GPU: argument checks and their messages, in the order of the reference's host wrappers
(src/nanoquant/kernel/cuda/gemm.cpp:36-98, gemv_kernel.cu:308-346), and what happens where it is not built."""
import pytest
import torch

from nanoquant_amd import _lib, ops

F16 = lambda *s: torch.zeros(*s, dtype=torch.float16)
I32 = lambda *s: torch.zeros(*s, dtype=torch.int32)


def _term(**other):
    args = dict(weight_u=I32(32, 128), weight_v=I32(16, 64), scale_g=F16(512), scale_l=F16(256), scale_h=F16(128), workspace=I32(64))
    args.update(other)
    return tuple(args.values())


# what is wrong, the message; on CPU tensors a call in order ends at the device check
@pytest.mark.parametrize("x,term,message", [
    (torch.zeros(5, 512), _term(), "Unsupported dtype: Marlin only supports Half and BFloat16"),
    (F16(5, 500), _term(), "k dimension mismatch"),
    (F16(5, 512), _term(scale_g=F16(511)), "s_in size mismatch"),
    (F16(5, 512), _term(scale_l=F16(255)), "s_out size mismatch"),
    (F16(5, 512), _term(workspace=I32(63)), "workspace too small"),
    (F16(5, 512), _term(), "x must be a CUDA tensor"),
])
def test_prefill_checks(x, term, message):
    for call in (lambda: ops.marlin_nanoquant_forward(x, *term), lambda: ops.gemm_forward_with_bias(x, *term, None), lambda: ops.gemm_group_forward(x, [term]),
                 lambda: ops.gemm_group_sum_forward(x, [[term]])):
        with pytest.raises(RuntimeError, match=message):
            call()


@pytest.mark.parametrize("x,other,message", [
    (torch.zeros(5, 512), {}, "Unsupported dtype"), (F16(5, 500), {}, "k dimension mismatch"), (F16(5, 512), {"scale_h": F16(255)}, "s_out size mismatch"),
    (F16(5, 512), {}, "x must be a CUDA tensor"),
])
def test_single_matrix_checks(x, other, message):
    args = dict(weight=I32(32, 128), scale_g=F16(512), scale_h=F16(256), workspace=I32(64))
    with pytest.raises(RuntimeError, match=message):
        ops.marlin_onebit_forward(x, **{**args, **other})


@pytest.mark.parametrize("call", [
    lambda x, t: ops.gemm_group_forward([x], [t, t]),
    lambda x, t: ops.gemm_group_forward(x, [t], biases=[None, None]),
    lambda x, t: ops.gemm_group_forward(x, [t], outs=[]),
    lambda x, t: ops.gemm_group_sum_forward([x], [[t], [t]]),
    lambda x, t: ops.gemm_group_sum_forward([x], [[]]),
])
def test_lists_of_different_lengths(call):
    with pytest.raises(RuntimeError, match=r"one x (and at least one term per weight|\(and one bias / output entry\) per term)"):
        call(F16(5, 512), _term())


def test_empty_groups():
    assert ops.gemm_group_forward(F16(5, 512), []) == [] and ops.gemm_group_sum_forward(F16(5, 512), []) == []


def test_terms_that_are_no_terms():
    with pytest.raises(ValueError, match="a term is"):
        ops.gemm_group_forward(F16(5, 512), [_term()[:5]])
    with pytest.raises(TypeError, match="weight_v must be a tensor"):
        ops.gemm_group_forward(F16(5, 512), [(I32(32, 128), 3, None, None, None, I32(64))])


def test_decode_checks_in_order():
    args = (F16(1, 64), F16(64), I32(32, 2), None, I32(96, 1), F16(96))
    with pytest.raises(RuntimeError, match="Support only Half or BFloat16"):
        ops.gemv_forward_with_bias(torch.zeros(1, 64), *args[1:], None)
    with pytest.raises(RuntimeError, match="x must be a CUDA tensor"):
        ops.gemv_forward_with_bias(*args, None)


def test_a_missing_build_is_an_import_error():
    broken = ops._Unbuilt(ImportError("not there"))
    with pytest.raises(ImportError, match="not there"):
        broken.gemm_group([], [])
    assert _lib.host().__name__ == "nanoquant_amd._host"


def test_no_panel_without_need():
    # argument checks only: no device is asked
    lib = _lib.lib()
    assert lib.nq_gemm_group_wants_panel(None, 1, 128, 0) == 0
    arr = (ops.NqGemmTerm * 1)(ops.NqGemmTerm(*[None] * 9, 512, 256, 128))
    assert lib.nq_gemm_group_wants_panel(arr, 1, 128, 2) == 0 and lib.nq_gemm_group_wants_panel(arr, 1, 0, 1) == 0
    assert lib.nq_gemm_group_wants_panel(arr, 1, 128, 1) == 1


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,r,m", [(512, 256, 0), (512, 0, 128), (-256, 256, 128), (512, 256, 100), (500, 256, 128), (512, 300, 128)])
def test_no_panel_for_sizes_that_are_refused(n, r, m, mode):
    good, bad = (ops.NqGemmTerm(*[None] * 9, *sizes) for sizes in ((512, 256, 128), (n, r, m)))
    assert _lib.lib().nq_gemm_group_wants_panel((ops.NqGemmTerm * 2)(good, bad), 2, 128, mode) == 0


# tokens, n, r, m; whether a stage can be a panel launch (32-bit offsets into x, h, y and the signs)
@pytest.mark.parametrize("tokens,n,r,m,fits", [
    (100000, 28672, 28672, 28672, 0),                        # 5.7 GB of x, h and y
    (64, 2 ** 25, 256, 32, 1), (64, 2 ** 25, 2 ** 25, 32, 0),     # 4 GiB of x; of h as well
    (64, 2 ** 25 - 256, 256, 32, 1),
    (33, 2 ** 25, 2 ** 25, 32, 0),                           # in whole token blocks
    (1, 2 ** 22, 2 ** 18, 2 ** 18, 0),                       # signs of 128 and 8 GiB
])
def test_panels_only_where_their_offsets_reach(tokens, n, r, m, fits):
    arr = (ops.NqGemmTerm * 1)(ops.NqGemmTerm(*[None] * 9, n, r, m))
    assert _lib.lib().nq_gemm_group_wants_panel(arr, 1, tokens, 1) == fits


def test_chains_of_terms_that_are_none():
    import ctypes
    term = lambda h, y, m=64, s_in=None: ops.NqGemmTerm(4096, 4096, 4096, s_in, None, None, None, h, y, 256, 256, m)
    call = lambda terms, nxt: _lib.lib().nq_gemm_nanoquant_sum((ops.NqGemmTerm * len(terms))(*terms), (ctypes.c_int * len(nxt))(*nxt), len(terms), 5, 0,
                                                               None, 0, 0, None)
    null, shape = -2, -3                                                                   # NQ_ERR_NULL, NQ_ERR_SHAPE
    for terms, nxt in [([term(16, 32), term(48, None)], [0, -1]),                          # a term behind itself
                       ([term(16, 32), term(48, None)], [2, -1]),                          # past the end
                       ([term(16, 32), term(48, None, m=96)], [1, -1]),                    # other rows
                       ([term(16, 32), term(48, 64), term(80, None)], [2, 2, -1]),         # one term in two chains
                       ([term(16, 32), term(48, 32)], [-1, -1]),                           # one output twice
                       ([term(16, 32), term(48, None, s_in=4096)], [1, -1])]:              # two kernels
        assert call(terms, nxt) == shape, nxt
    assert call([term(16, 32), term(48, None)], [-1, -1]) == null               # a first term without y


def test_no_workspace_is_made_while_a_graph_is_captured(monkeypatch):
    # it would hold whatever was there until the graph runs, and calls outside the graph would use it
    import contextlib
    import types
    made, capturing = [], [True]
    monkeypatch.setattr(ops, "_panel_ws_cache", {})
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(cuda_stream=7))
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(_lib, "lib", lambda: types.SimpleNamespace(nq_gemm_panel_workspace_bytes=lambda: 256))
    monkeypatch.setattr(torch, "zeros", lambda n, **kw: made.append(n) or torch.empty(n))
    device = torch.device("cuda", 0)
    assert ops._panel_workspace(device) is None and not made and not ops._panel_ws_cache
    capturing[0] = False
    buf = ops._panel_workspace(device)
    assert made == [256]
    capturing[0] = True
    assert ops._panel_workspace(device) is buf and made == [256]
