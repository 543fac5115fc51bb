"""Grouped prefill above 160 tokens: both sides of the lines between few-token tiles, block tiles and panels."""
import numpy as np
import pytest
import torch

from nanoquant_amd import ops, packing
from oracle import nq_oracle as oracle

pytestmark = pytest.mark.gpu


# (tokens, n, r, m): 64-token x 128-row block workgroups of the two GEMMs in the comments
@pytest.mark.parametrize("tokens,n,r,m", [
    (161, 4096, 256, 320),       # 6 and 9: few-token tiles (16 k tiles), block tiles (one)
    (384, 1792, 4096, 512),      # 192 on 7 k tiles: the last one on few-token tiles; 24 on 16
    (384, 1792, 4352, 256),      # 204: block tiles
    (384, 4096, 7680, 288),      # 360 on 16 k tiles: the last one on few-token tiles
    (330, 4096, 7936, 288),      # 372: panels or block tiles; 18 on 31 k tiles
    (450, 11008, 1280, 256),     # 80 on 43 k tiles: few-token tiles
    (450, 11008, 1536, 256),     # 96: panels
    (500, 256, 4096, 1536),      # second GEMM, 96 on 16 k tiles: the last one on few-token tiles at 401 to 512 tokens
    (500, 256, 4096, 1664),      # 104: block tiles
    (1500, 4096, 512, 256),      # 96 on 16 k tiles: the last one on few-token tiles above 1280 tokens
    (1800, 4096, 256, 256),      # 58 above 1536: block tiles
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_either_side_of_the_lines(dev, dtype, tokens, n, r, m):
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(dtype)
    f32 = lambda t: t.float().cpu().numpy()
    vt, u, s_in, s_mid, s_out = oracle.synth_term(m, n, r, 9500)
    sc = (to(s_in), to(s_mid), to(s_out))
    packed = packing.marlin_nanoquant_packer(torch.from_numpy(vt).T.contiguous().to(dev), torch.from_numpy(u).T.contiguous().to(dev), *sc)
    x = to(oracle.synth_x(tokens, n, 9501))
    ref = oracle.layer_forward(f32(x), vt, u, *(f32(s) for s in sc))
    for panel in ("auto", "never"):
        y = ops.gemm_group_forward([x], [packed], panel=panel)[0]
        torch.cuda.synchronize()
        err = oracle.max_rel_err(f32(y), ref)
        print(f"group {tokens} tokens {n}->{r}->{m} {dtype} panel={panel}: {err:.2e}", flush=True)
        # h and the result are rounded to the 16-bit type: half an ulp each, 2^-11 (fp16) or 2^-8 (bf16), of values near the largest
        assert err < 3 * (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8), (panel, err)
    assert ops.panel_status(dev) == 0


# (tokens, (n, r, m) of a linear, of a neighbour that puts the launch beyond the few-token tiles)
@pytest.mark.parametrize("tokens,linear,neighbour", [
    (3072, (4096, 256, 256), (4096, 2048, 256)),     # few rows at many tokens: 96 block workgroups on 16 k tiles
    (512, (256, 4096, 3072), (256, 4096, 8192)),     # a second GEMM: 192 on 16 k tiles
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_block_tiles_where_few_token_tiles_are_slower(dev, dtype, tokens, linear, neighbour):
    # the route shows in the bits: block tiles add the k tiles one behind the other, few-token tiles in four shares
    gen = torch.Generator(device=dev)
    gen.manual_seed(11)
    signs = lambda a, b: torch.randint(0, 2, (a, b), dtype=torch.int8, device=dev, generator=gen) * 2 - 1
    scale = lambda k: (torch.rand(k, device=dev, generator=gen) + 0.01).to(dtype)
    terms = [packing.marlin_nanoquant_packer(signs(n, r), signs(r, m), scale(n), scale(r), scale(m)) for n, r, m in (linear, neighbour)]
    x = torch.randn(tokens, linear[0], device=dev, generator=gen).to(dtype)
    print(f"group {tokens} tokens {linear} beside {neighbour} {dtype}", flush=True)
    alone = ops.gemm_group_forward([x], terms[:1], panel="never")[0]
    beside = ops.gemm_group_forward([x, x], terms, panel="never")[0]
    torch.cuda.synchronize()
    assert torch.equal(alone, beside)


# (tokens, linears [(n, r, m)]): a first GEMM of 43, a second one of 16 k tiles beside ones of 4 and 6
@pytest.mark.parametrize("tokens,linears", [
    (256, [(11008, 1024, 256), (1024, 1024, 256)]),
    (333, [(256, 4096, 512), (256, 1536, 1024), (256, 1536, 1024)]),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_the_longest_k_of_a_group_decides(dev, dtype, tokens, linears):
    # the one of the long k gets the bits it gets alone: few-token tiles in both calls
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(dtype)
    f32 = lambda t: t.float().cpu().numpy()
    packed, xs, refs = [], [], []
    for i, (n, r, m) in enumerate(linears):
        vt, u, *scales = oracle.synth_term(m, n, r, 9600 + i)
        sc = [to(s) for s in scales]
        packed.append(packing.marlin_nanoquant_packer(torch.from_numpy(vt).T.contiguous().to(dev), torch.from_numpy(u).T.contiguous().to(dev), *sc))
        xs.append(to(oracle.synth_x(tokens, n, 9610 + i)))
        refs.append(oracle.layer_forward(f32(xs[-1]), vt, u, *(f32(s) for s in sc)))
    print(f"mixed group {tokens} tokens {linears} {dtype}", flush=True)
    alone = ops.gemm_group_forward(xs[:1], packed[:1])[0]
    together = ops.gemm_group_forward(xs, packed)
    torch.cuda.synchronize()
    assert torch.equal(alone, together[0])
    for y, ref in zip(together, refs):
        # h and the result are rounded to the 16-bit type, as above
        assert oracle.max_rel_err(f32(y), ref) < 3 * (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8)
    assert ops.panel_status(dev) == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_inputs_of_their_own_count_by_themselves(dev, dtype):
    # six linears of 256 rows on 640 tokens: few-token tiles on one input (the bits of one of them alone), block tiles on six
    # inputs (the bits beside a neighbour that fills the device)
    gen = torch.Generator(device=dev)
    gen.manual_seed(12)
    signs = lambda a, b: torch.randint(0, 2, (a, b), dtype=torch.int8, device=dev, generator=gen) * 2 - 1
    scale = lambda k: (torch.rand(k, device=dev, generator=gen) + 0.01).to(dtype)
    make = lambda r: packing.marlin_nanoquant_packer(signs(4096, r), signs(r, 256), scale(4096), scale(r), scale(256))
    terms, big = [make(256) for _ in range(6)], make(8192)
    xs = [torch.randn(640, 4096, device=dev, generator=gen).to(dtype) for _ in range(6)]
    print(f"six linears on one input and on six {dtype}", flush=True)
    run = lambda x, t: ops.gemm_group_forward(x, t, panel="never")
    few, block = run(xs[:1], terms[:1])[0], run([xs[0], xs[0]], [terms[0], big])[0]
    one, six = run([xs[0]] * 6, terms)[0], run(xs, terms)[0]
    torch.cuda.synchronize()
    assert torch.equal(one, few) and torch.equal(six, block) and not torch.equal(few, block)


# (tokens, weights as lists of (n, r, m)): the second GEMMs differ in k, and panels are estimated a little ahead of tiles, too little to
# be taken.  us apart on tiles / apart on panels / as sums
@pytest.mark.parametrize("tokens,weights", [
    (655, [[(8960, 3328, 12288), (8960, 3072, 12288)], [(8960, 3840, 5408)]]),      # 241 / 237 / 223
    (868, [[(6656, 3584, 12768), (6656, 3840, 12768)]]),                           # 234 / 237 / 228
    (1037, [[(1792, 3584, 4384), (1792, 2560, 4384)], [(1792, 3840, 7072)]]),       # 151 / 153 / 148
])
def test_sums_are_compared_with_the_launch_that_would_be_made(dev, tokens, weights):
    import ctypes

    from nanoquant_amd import _lib
    flat = [(w, t) for w, terms in enumerate(weights) for t in range(len(terms))]
    follows = [flat.index((w, t + 1)) if (w, t + 1) in flat else -1 for w, t in flat]
    arr = (ops.NqGemmTerm * len(flat))(*[ops.NqGemmTerm(4096, 4096, 4096, 4096, None, None, None, 4096 * (i + 1), 16 * (i + 1), *weights[w][t])
                                         for i, (w, t) in enumerate(flat)])
    assert _lib.lib().nq_gemm_sum_pays(arr, (ctypes.c_int * len(flat))(*follows), len(flat), tokens) == 1      # a question, no launch


# (tokens, linears (n, r, m), whether a stage is a panel launch); us on tiles / with the first stage on panels / the second
@pytest.mark.parametrize("tokens,linears,panel", [
    (1280, [(4096, 2048, 4096), (12288, 3072, 4096)], 1),      # k of 16 and 48 tiles: 196 / 167 / 202
    (640, [(4096, 2048, 4096), (12288, 3072, 4096)], 1),       # 115 / 103 / 117
    (640, [(4096, 1536, 4096), (11008, 2304, 4096)], 1),       # 90 / 85 / 94
    (1536, [(1024, 2048, 4096), (1024, 3072, 12288), (1024, 3072, 12288)], 0),      # k of 8 and 12 tiles: tiles ahead by 5 %
    (256, [(4096, 2048, 4096)] * 4 + [(4096, 3072, 11008)] * 2 + [(11008, 3072, 4096)], 1),      # 119 / 111
    (768, [(4096, 2048, 4096)] * 4 + [(4096, 3072, 11008)] * 2 + [(11008, 3072, 4096)], 0),      # 264 / 272
    (1024, [(4096, 2048, 4096)] * 4 + [(4096, 3072, 11008)] * 2 + [(11008, 3072, 4096)], 0),     # 347 / 357
    (40, [(8192, 4096, 8192), (8192, 1024, 1024), (8192, 1024, 1024), (28672, 6400, 8192)], 0),     # 16 workgroups to a panel: 51 / 67
    (99, [(8192, 2560, 8192), (28672, 3840, 8192)], 0),        # 60 / 76
])
def test_panels_beside_tiles_where_k_differs(dev, tokens, linears, panel):
    from nanoquant_amd import _lib
    # inputs by width, h by linear, as a group call has them
    arr = (ops.NqGemmTerm * len(linears))(*[ops.NqGemmTerm(n, 4096, 4096, 4096, None, None, None, 4096 * (i + 1), 16 * (i + 1), n, r, m)
                                           for i, (n, r, m) in enumerate(linears)])
    assert _lib.lib().nq_gemm_group_wants_panel(arr, len(linears), tokens, 0) == panel      # a question, no launch
