"""Long run lists at batch 8 and 16 in tile order (one-bit fp4 weights x fp6 pieces of the input) against the oracle."""
import numpy as np
import pytest
import torch

from nanoquant_amd import DecodeRunList, packing
from oracle import nq_oracle as oracle

pytestmark = pytest.mark.gpu

# (m, n, r): whole and cut row pairs, words that are no multiple of four, K % 8 != 0, inputs of one chunk (32 units at batch
# 16, 64 at batch 8: exactly, one over) and of several, and a second stage that is one column group over a chunk
SHAPES = [(520, 1504, 416), (96, 160, 64), (1000, 1100, 333), (64, 4100, 96), (256, 8200, 4096), (300, 12000, 4128), (512, 8192, 928)]
# Three roundings to the nearest fp6 number leave at most 2^-13.9 of a unit's largest value per element: 1e-4 of a sum of random
# signs over two stages, one sigma, against a largest of many that is 4 to 5 sigma itself; 16-bit outputs add half an ulp.
F32_TOL = 3e-4
TOL = {torch.float16: F32_TOL + 2.0 ** -11, torch.bfloat16: F32_TOL + 2.0 ** -8}


def _filled_list(dev, batch, dtype, copies, seed, **kw):
    """A list long enough for the fp6 kernel: `copies` linears of 6400 x 28672 and 8192 x 6400 random signs on one input."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    m, n, r = 8192, 28672, 6400
    word = lambda rows, cols: torch.randint(-2 ** 31, 2 ** 31 - 1, (rows, cols // 32), dtype=torch.int32, device=dev, generator=gen)
    scale = lambda k: (torch.rand(k, device=dev, generator=gen) * 0.02 + 1e-3).to(dtype)
    v, u, sc = word(r, n), word(m, r), (scale(n), scale(r), scale(m))
    x = torch.randn(batch, n, device=dev, generator=gen).to(dtype)
    rl = DecodeRunList(batch, dtype, dev, **kw)
    vt, ut = packing.tile_words(v), packing.tile_words(u)
    return rl, lambda: rl.add(x, sc[0], vt, sc[1], ut, sc[2], tiled=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch", [8, 16])
def test_long_tile_order_lists(dev, batch, dtype):
    rl, filler = _filled_list(dev, batch, dtype, 10, 5)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(dtype)
    f64 = lambda t: t.float().cpu().numpy().astype(np.float64)
    pack = lambda w: packing.tile_words(packing.binary_packer(torch.from_numpy(w), "half2").to(dev))
    fillers, checked = [filler()], []
    for i, (m, n, r) in enumerate(SHAPES):
        vt, u, s_in, s_mid, s_out = oracle.synth_term(m, n, r, 9000 + i)
        vt_p, u_p, mid_p = oracle.pad_rank(vt, u, s_mid, 32)
        x, sc = to(oracle.synth_x(batch, n, 9100 + i)), (to(s_in), to(mid_p), to(s_out))
        ref = oracle.layer_forward(f64(x), vt, u, f64(sc[0]), f64(to(s_mid)), f64(sc[2]), dtype=np.float64)
        args = (x, sc[0], pack(vt_p), sc[1], pack(u_p), sc[2])
        bias = to(np.linspace(-1, 1, m, dtype=np.float32) * np.abs(ref).max()) if i % 2 else None
        with_bias = ref + (f64(bias) if bias is not None else 0.0)
        checked.append((rl.add(*args, tiled=True, bias=bias), with_bias, TOL[dtype]))
        # the same as an fp32 result, and a third time added onto that one
        first = rl.add(*args, tiled=True, out_f32=True)
        checked.append((first, ref, F32_TOL))
        checked.append((rl.add(*args, tiled=True, out_f32=True, addend=rl.outputs[first], y_from=first), 2 * ref, F32_TOL))
        fillers.append(filler())
    while len(fillers) < 10:
        fillers.append(filler())
    ys = rl.run()
    torch.cuda.synchronize()
    print(f"fp6 list batch={batch} {dtype}: plan flags {rl._plan.bound:#x}", flush=True)
    assert rl.status() == 0 and rl._plan.bound & 64
    for k, ref, tol in checked:
        err = oracle.max_rel_err(ys[k].float().cpu().numpy(), ref)
        assert err < tol, (SHAPES[k // 4] if k else None, k, err)
    # every row is summed by one wavefront in the order of its columns, wherever the slices are cut and in every launch
    base = [y.clone() for y in ys]
    assert all(torch.equal(base[fillers[0]], base[k]) for k in fillers)
    for rep in range(3):
        again = rl.run()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(base, again)), rep


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch", [8, 16])
def test_long_lists_compute_exactly_on_the_fp6_pieces(dev, batch, dtype):
    # The oracle's restatement of the staging predicts the output up to the fp32 sums and the few elements of h that an fp32
    # rounding moves to the next step of their unit (2^-11.9 of its maximum, one of hundreds that are added; 5e-8 measured): a
    # lost piece (4e-3), one of another size (3e-4), a wrong column or block scale (O(1)) cannot hide in the tolerance.  Batch row 1 has channels 1000 times the rest.
    m, n, r = 768, 1504, 416                                       # 47 and 13 words per row
    vt, u, s_in, s_mid, s_out = oracle.synth_term(m, n, r, 9400)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(dtype)
    f64 = lambda t: t.float().cpu().numpy().astype(np.float64)
    pack = lambda w: packing.tile_words(packing.binary_packer(torch.from_numpy(w), "half2").to(dev))
    x = oracle.synth_x(batch, n, 9401)
    x[1, [3, 700, 701]] *= 1000
    rl, filler = _filled_list(dev, batch, dtype, 10, 8)
    xd, sc = to(x), (to(s_in), to(s_mid), to(s_out))
    k = rl.add(xd, sc[0], pack(vt), sc[1], pack(u), sc[2], tiled=True, out_f32=True)
    for _ in range(9):
        filler()
    y = f64(rl.run()[k])
    assert rl.status() == 0 and rl._plan.bound & 64
    a, b, c = (f64(t) for t in sc)
    for shifts, close in (((0, 4, 9), True), ((0, 4), False), ((0, 4, 8), False)):
        stage = lambda v, signs: oracle.staged_input_fp6(v, shifts=shifts) @ signs.T.astype(np.float64)
        ref = stage((stage(f64(xd) * a, vt) * b).astype(np.float32).astype(np.float64), u) * c
        err = (np.abs(y - ref).max(axis=1) / np.abs(ref).max(axis=1)).max()
        print(f"fp6 staging batch={batch} {dtype} pieces {shifts}: {err:.2e}", flush=True)
        assert (err < 2e-5) == close, (shifts, err)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("batch", [8, 16])
def test_outlier_channels_cost_no_more_than_16_bit_operands(dev, batch, dtype):
    """Four input channels 1000 times the rest, judged against the share of the ordinary channels, with what rounding x * s_in
    and h to 16 bits costs on the same input as the yardstick (the 16-bit operands make both).  The units of the outliers keep 5
    bits of their ordinary channels; the sums, which the outliers' own rounding dominates, are closer than with 16 bits."""
    m, n, r = 1024, 4096, 512
    vt, u, s_in, s_mid, s_out = oracle.synth_term(m, n, r, 510)
    x = oracle.synth_x(batch, n, 511)
    hot = [5, 1300, 2049, 4000]
    x[:, hot] = (x[:, hot] * 1000.0).astype(x.dtype)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(dtype)
    f64 = lambda t: t.float().cpu().numpy().astype(np.float64)
    pack = lambda w: packing.tile_words(packing.binary_packer(torch.from_numpy(w), "half2").to(dev))
    rounded = lambda v: torch.from_numpy(v).to(dtype).double().numpy()
    for pow2 in (False, True):                                     # with s_in = 2^-7, x * s_in fits 16 bits: only h is rounded
        xd, sc = to(x), (to(np.full(n, 2.0 ** -7)) if pow2 else to(s_in), to(s_mid), to(s_out))
        rl, filler = _filled_list(dev, batch, dtype, 10, 9)
        filler()
        k = rl.add(xd, sc[0], pack(vt), sc[1], pack(u), sc[2], tiled=True, out_f32=True)
        for _ in range(9):
            filler()
        y = f64(rl.run()[k])
        assert rl.status() == 0 and rl._plan.bound & 64
        xe, (a, b, c) = f64(xd), (f64(t) for t in sc)
        ref = oracle.layer_forward(xe, vt, u, a, b, c, dtype=np.float64)
        calm = xe.copy()
        calm[:, hot] = 0.0
        rest = oracle.layer_forward(calm, vt, u, a, b, c, dtype=np.float64)
        h = (rounded(xe * a) @ vt.T.astype(np.float64)) * b
        ref16 = (rounded(h) @ u.T.astype(np.float64)) * c
        floor = 0.1 * np.sqrt(np.mean(rest * rest))
        rms = lambda d: float(np.sqrt(np.mean((d / (np.abs(rest) + floor)) ** 2)))
        print(f"fp6 outliers batch={batch} {dtype} pow2={pow2}: {rms(y - ref):.3e} (16 bits: {rms(ref16 - ref):.3e})", flush=True)
        assert rms(y - ref) <= rms(ref16 - ref)


@pytest.mark.parametrize("batch", [8, 16])
def test_a_batch_row_that_is_not_finite_stays_alone(dev, batch):
    rl, filler = _filled_list(dev, batch, torch.bfloat16, 9, 6)
    vt, u, s_in, s_mid, s_out = oracle.synth_term(160, 1024, 256, 9200)
    to = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(torch.bfloat16)
    pack = lambda w: packing.tile_words(packing.binary_packer(torch.from_numpy(w), "half2").to(dev))
    x = to(oracle.synth_x(batch, 1024, 9201))
    k = rl.add(x, to(s_in), pack(vt), to(s_mid), pack(u), to(s_out), tiled=True, out_f32=True)
    for _ in range(9):
        filler()
    clean = rl.run()[k].clone()
    assert rl._plan.bound & 64 and torch.isfinite(clean).all()
    keep = x.clone()
    for row, value in ((3, float("inf")), (batch - 1, float("nan")), (0, -float("inf"))):
        x.copy_(keep)
        x[row, 777] = value
        y = rl.run()[k]
        torch.cuda.synchronize()
        others = [b for b in range(batch) if b != row]
        assert torch.isnan(y[row]).all() and torch.equal(y[others], clean[others]), (row, value)
    x.copy_(keep)
    x[5] = 0                                                       # a row of zeros, and one far below the others
    x[6] *= 2.0 ** -60
    y = rl.run()[k]
    torch.cuda.synchronize()
    assert rl.status() == 0 and (y[5] == 0).all() and torch.equal(y[6], clean[6] * 2.0 ** -60)


@pytest.mark.parametrize("batch", [8, 16])
def test_long_lists_with_a_row_major_linear_keep_the_16_bit_operands(dev, batch):
    rl, filler = _filled_list(dev, batch, torch.float16, 9, 7)
    for _ in range(9):
        filler()
    vt, u, s_in, s_mid, s_out = oracle.synth_term(160, 1024, 256, 9300)
    f = lambda a: torch.from_numpy(a).to(dev)
    words = lambda w: packing.binary_packer(torch.from_numpy(w), "half2").to(dev)
    x = oracle.synth_x(batch, 1024, 9301)
    k = rl.add(f(x), f(s_in), words(vt), f(s_mid), words(u), f(s_out))
    y = rl.run()[k]
    torch.cuda.synchronize()
    assert rl.status() == 0 and not rl._plan.bound & 64
    ref = oracle.layer_forward(x.astype(np.float64), vt, u, s_in, s_mid, s_out, dtype=np.float64)
    assert oracle.max_rel_err(y.float().cpu().numpy(), ref) < 1e-3
