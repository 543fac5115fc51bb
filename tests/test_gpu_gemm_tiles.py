"""Prefill tiles at their edges: every tile size of csrc/nq_gemm.hip with ragged tokens and rows, k of one tile up to more than
the ring and the k groups hold, against the dense definition in 64 bits (src/nanoquant/modules/linear.py:248-257 of the
reference)."""
import numpy as np
import pytest
import torch

from nanoquant_amd import ops, packing
from oracle import nq_oracle as oracle
from test_tile_choice import ALONE, sum_route, tile

pytestmark = pytest.mark.gpu
# half an ulp of the 16-bit result, and as much again for the h that feeds the second GEMM
ROUND = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _onebit(dev, tokens, k, rows, dtype, scaled, seed):
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    signs = torch.randint(0, 2, (rows, k), dtype=torch.int8, device=dev, generator=gen) * 2 - 1
    scale = lambda n: (torch.rand(n, device=dev, generator=gen) + 0.01).to(dtype)
    s_in, s_out = scale(k) if scaled else None, scale(rows)
    bits, si, so, words = packing.marlin_onebit_packer(signs, s_in, s_out)
    x = torch.randn(tokens, k, device=dev, generator=gen).to(dtype)
    xs = x.double() * (s_in.double() if scaled else 1.0)
    return x, bits, si, so, torch.zeros(max(words, 1), dtype=torch.int32, device=dev), (xs @ signs.double().T) * s_out.double()


# (tokens, k, rows), the tile with and without input scales: 32 x 32 up to 32 x 96 split k four ways (k tiles left over for none, one,
# three of the four wavefronts), 64 x 128 up to 128 x 256 do not
@pytest.mark.parametrize("tokens,k,rows,tiles", [
    (1, 256, 32, "32x32"), (31, 512, 64, "32x32"), (33, 1280, 96, "32x32"), (65, 2304, 160, "32x32"),      # 1, 2, 5, 9 k tiles
    (128, 4096, 3104, "32x64"), (200, 1792, 2080, "32x64"), (250, 2048, 3136, "32x64"),      # a row tile left over, the same, none
    (161, 2816, 3072, "32x96"), (200, 2816, 3104, "32x96"), (250, 2048, 2080, "32x96"),      # none, one and two row tiles left over
    (333, 4096, 3104, "32x96 64x128"),
    (333, 1024, 3168, "64x128"), (700, 256, 2080, "64x128"), (193, 2560, 8224, "64x128"), (4097, 256, 8224, "64x128"),
    (400, 768, 16416, "64x256"), (250, 512, 8224, "64x256"), (2049, 2048, 4128, "64x256"),
    (1000, 1280, 4128, "128x256"), (2049, 512, 12320, "128x256"),
    (352, 1024, 3168, "64x128"), (353, 1024, 3168, "64x128"), (2112, 512, 12320, "128x256"), (2113, 512, 12320, "128x256"),   # half a tile of tokens left, one more
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("scaled", [True, False])
def test_tiles_at_their_edges(dev, tokens, k, rows, tiles, dtype, scaled):
    assert "%dx%d" % tile(ALONE, tokens, [k], [rows], scaled) == tiles.split()[0 if scaled else -1]
    x, bits, si, so, workspace, ref = _onebit(dev, tokens, k, rows, dtype, scaled, tokens + k)
    print(f"tile {tokens} tokens {k} -> {rows} {dtype} scaled={scaled}", flush=True)
    y = torch.ops.binary_kernels.marlin_onebit_forward(x, bits, si, so, workspace)
    torch.cuda.synchronize()
    err = ((y.double() - ref).abs().max() / ref.abs().max()).item()
    assert err < 1.2 * ROUND[dtype], err                     # products are exact, sums are fp32: the rounding of the result


@pytest.mark.parametrize("tokens", [5, 200])
def test_output_scales_that_begin_anywhere(dev, tokens):
    # of one linear by itself, on few-token and on block tiles: slices at every element offset give the bits of an aligned scale
    x, bits, si, so, workspace, _ = _onebit(dev, tokens, 512, 2080, torch.float16, True, 8)
    want = torch.ops.binary_kernels.marlin_onebit_forward(x, bits, si, so, workspace)
    for offset in range(1, 8):
        own = torch.full((offset + so.numel() + 8,), float("nan"), dtype=so.dtype, device=dev)[offset:offset + so.numel()]
        own.copy_(so)
        print(f"scale at element {offset}, {tokens} tokens", flush=True)
        y = torch.ops.binary_kernels.marlin_onebit_forward(x, bits, si, own, workspace)
        torch.cuda.synchronize()
        assert torch.equal(y, want), offset


@pytest.mark.parametrize("scaled", [True, False])
def test_more_columns_than_a_tile_of_tokens_can_address(dev, scaled):
    # token by token, 16 to a launch
    tokens, k, rows, dtype = 18, 2 ** 22 + 256, 256, torch.float16
    x, bits, si, so, workspace, ref = _onebit(dev, tokens, k, rows, dtype, scaled, 9)
    print(f"{k} columns scaled={scaled}", flush=True)
    y = torch.ops.binary_kernels.marlin_onebit_forward(x, bits, si, so, workspace)
    torch.cuda.synchronize()
    err = ((y.double() - ref).abs().max() / ref.abs().max()).item()
    assert err < 1.2 * ROUND[dtype], err
    # in a group beside an ordinary linear: the bits that both get by themselves
    x2, bits2, si2, so2, _, _ = _onebit(dev, tokens, 512, rows, dtype, scaled, 10)
    out = _onebit(dev, 1, rows, 64, dtype, False, 11)[1]
    terms = [(bits, out, si, so, None, workspace), (bits2, out, si2, so2, None, workspace)]
    alone = [torch.ops.binary_kernels.marlin_nanoquant_forward(a, *t) for a, t in zip((x, x2), terms)]
    group = ops.gemm_group_forward([x, x2], terms, panel="never")
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(alone, group))


@pytest.mark.parametrize("tokens", [100, 128, 160])
def test_other_tiles_for_many_rows_below_160_tokens(dev, tokens):
    # 2 x 8192 rows over a short rank: block tiles where the group may take any, the bits of the linear alone where it may not
    dtype, n = torch.float16, 512
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(dtype)
    packed, refs = [], []
    x = f(oracle.synth_x(tokens, n, 5))
    for i in range(2):
        vt, u, *scales = oracle.synth_term(8192, n, 512, 70 + i)
        sc = [f(s) for s in scales]
        packed.append(packing.marlin_nanoquant_packer(torch.from_numpy(vt).T.contiguous().to(dev), torch.from_numpy(u).T.contiguous().to(dev), *sc))
        refs.append(oracle.layer_forward(x.float().cpu().numpy(), vt, u, *(s.float().cpu().numpy() for s in sc)))
    print(f"many rows {tokens} tokens", flush=True)
    alone = [torch.ops.binary_kernels.marlin_nanoquant_forward(x, *p) for p in packed]
    same, free = ops.gemm_group_forward(x, packed, panel="never"), ops.gemm_group_forward(x, packed)
    torch.cuda.synchronize()
    for a, s, y, ref in zip(alone, same, free, refs):
        assert torch.equal(a, s)
        assert oracle.max_rel_err(y.float().cpu().numpy(), ref) < 3 * ROUND[dtype]


# Sums of terms: chains of 1 to 3 terms of uneven rank, ranks of one tile up to many, a bias on some terms; every tile that sums
# (32 x 32, 32 x 64 and 32 x 96 with k split, 64 x 128, 64 x 256) with tokens and rows left over.
@pytest.mark.parametrize("tokens,spec,tiles", [
    (1, [(32, (200, 100)), (96, (512,))], "32x32"),
    (33, [(160, (256, 1280, 300)), (64, (100,)), (3104, (700, 256))], "32x32"),
    (70, [(3104, (1280, 300))], "32x64"), (157, [(2080, (512, 300))], "32x64"),
    (190, [(3104, (2304, 512))], "32x96"), (157, [(4128, (1280, 300))], "32x96"), (520, [(1056, (1280, 300))], "32x96"),
    (200, [(3104, (512, 2304)), (2080, (256,))], "64x128"),
    (333, [(3104, (256, 256, 768)), (1056, (2048, 100))], "64x128"),
    (700, [(4128, (300, 100)), (2080, (256,))], "64x128"),
    (1000, [(8224, (256, 256))], "64x128"),
    (992, [(8224, (256, 256))], "64x128"), (993, [(8224, (256, 256))], "64x128"),
    (157, [(8224, (1280, 512)), (8224, (1280, 512))], "64x256"), (1000, [(2080, (2304, 512))], "64x256"),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_sums_of_terms(dev, tokens, spec, tiles, dtype):
    f = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    host = lambda a: a.float().cpu().numpy()
    n = 512
    x = f(oracle.synth_x(tokens, n, tokens)).to(dtype)
    groups, biases, refs = [], [], []
    for w, (m, ranks) in enumerate(spec):
        packed, own, ref = [], [], 0.0
        for t, rank in enumerate(ranks):
            vt, u, *scales = oracle.synth_term(m, n, rank, 31 * tokens + 5 * w + t)
            sc = [f(s).to(dtype) for s in scales]
            bias = torch.linspace(-1, 1, m, device=dev).to(dtype) if (w + t) % 2 else None
            packed.append(packing.marlin_nanoquant_packer(f(vt).T.contiguous(), f(u).T.contiguous(), *sc))
            own.append(bias)
            ref = ref + oracle.layer_forward(host(x), vt, u, *(host(s) for s in sc)) + (0.0 if bias is None else host(bias))
        groups.append(packed)
        biases.append(own)
        refs.append(ref)
    size, pays = sum_route(tokens, [[(n, v.size(0) * 16, v.size(1) * 2) for _, v, *_ in terms] for terms in groups])
    assert "%dx%d" % size == tiles and pays
    print(f"sums {tokens} tokens {spec} {dtype}", flush=True)
    added, apart = ops.gemm_group_sum_forward(x, groups, biases), ops.gemm_group_sum_forward(x, groups, biases, panel="never")
    torch.cuda.synchronize()
    for y, z, ref in zip(added, apart, refs):
        err, err_apart = oracle.max_rel_err(host(y), ref), oracle.max_rel_err(host(z), ref)
        assert err < 3 * ROUND[dtype], err                   # h and the result are rounded, the sum is not
        assert err_apart < 5 * ROUND[dtype], err_apart       # and here every term's result and two additions
