"""The few-row decode kernel (csrc/nq_rows.hip) at the sizes where its split can go wrong: row blocks of 16 with a
remainder, one or two of them per workgroup, column chunks of 512 over one to eight (or four) wavefronts and several
rounds, rows of words that are not a multiple of four (the last unit of the last row is read from 16 bytes before the
end of the matrix), inputs without 16-byte alignment, and sums of terms; against the dense definition in fp64
(src/nanoquant/modules/linear.py:248-257 of the reference)."""
import numpy as np
import pytest
import torch

from nanoquant_amd import ops, packing
from oracle import nq_oracle as oracle

pytestmark = pytest.mark.gpu


def _cast(a, dtype):
    return torch.from_numpy(np.ascontiguousarray(a).astype(np.float32)).to(dtype)


def _eps(dtype):
    return 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8          # largest relative error of one rounding


def _close_in_norm(y, ref, dtype, roundings):
    """`roundings` roundings on the way (x * s_in, h, y) whose errors add up like a random walk over random signs."""
    d = y.double().cpu().numpy() - ref
    assert np.linalg.norm(d) <= np.sqrt(roundings) * _eps(dtype) * np.linalg.norm(ref)


def _close_in_every_element(y, ref, magnitude, dtype):
    """|error| <= eps (sum of the magnitudes of the rounded products) + eps |y|, and fp32 sums: 2^-24 per addition."""
    d = np.abs(y.double().cpu().numpy() - ref)
    assert (d <= magnitude * (_eps(dtype) + 2.0 ** -16) + 1.01 * _eps(dtype) * np.abs(ref)).all()


# rows: one row, a block and one row, 257 blocks (two per workgroup from 5 batch rows on), four wavefronts from 8192
# rows on; columns: part of a unit, 1, 2, 3 words over a unit, a chunk and one unit, 8 and 9 chunks, 17 chunks
@pytest.mark.parametrize("rows,cols", [(1, 8), (17, 32), (15, 40), (33, 160), (16, 512), (48, 640), (100, 96), (4100, 224),
                                       (70, 4096), (31, 4104), (40, 8480), (8192, 608), (8200, 2600)])
@pytest.mark.parametrize("batch", [1, 2, 3, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_stage(dev, dtype, batch, rows, cols):
    rng = np.random.default_rng(rows + 7 * cols + batch)
    signs = rng.integers(0, 2, size=(rows, cols), dtype=np.int8) * 2 - 1
    bits = packing.binary_packer(torch.from_numpy(signs), "half2").to(dev)
    x = _cast(rng.normal(size=(batch, cols)), dtype)
    s_col, s_row = (_cast(np.abs(rng.normal(0, 0.5, k)) + 0.1, dtype) for k in (cols, rows))
    print(f"rows stage {rows} x {cols} batch {batch} {dtype}", flush=True)
    f64 = lambda t: t.double().numpy()
    scaled = ops.gemv_stage_forward(x.to(dev), s_col.to(dev), bits, s_row.to(dev))
    plain = ops.gemv_stage_forward(x.to(dev), None, bits, None)
    torch.cuda.synchronize()
    xs, w = f64(x) * f64(s_col), signs.T.astype(np.float64)
    for y, ref, mag, roundings in ((scaled, xs @ w * f64(s_row), np.abs(xs).sum(1)[:, None] * f64(s_row), 2),
                                   # no rounded products here: 2^-23 of the magnitudes covers the fp32 additions
                                   (plain, f64(x) @ w, np.abs(f64(x)).sum(1)[:, None] * 2.0 ** -12, 1)):
        _close_in_every_element(y, ref, mag, dtype)
        if rows * batch >= 256 and cols >= 256:
            _close_in_norm(y, ref, dtype, roundings)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_inputs_without_16_byte_alignment(dev, dtype):
    # odd widths and a view that starts in the middle of 16 bytes give the same bits as an aligned copy
    rng = np.random.default_rng(3)
    for batch, rows, cols in ((1, 40, 1003), (4, 130, 517), (11, 64, 4097)):
        bits = packing.binary_packer(torch.from_numpy(rng.integers(0, 2, size=(rows, cols), dtype=np.int8) * 2 - 1), "half2").to(dev)
        pad = (cols + 31) // 32 * 32
        flat = _cast(rng.normal(size=batch * cols + 1), dtype).to(dev)
        x = flat[1:].view(batch, cols)                                    # 2 bytes off
        s_col = _cast(rng.normal(size=cols), dtype).to(dev)
        xa = torch.zeros(batch, pad, dtype=dtype, device=dev)
        xa[:, :cols] = x
        sa = torch.zeros(pad, dtype=dtype, device=dev)
        sa[:cols] = s_col
        print(f"unaligned rows stage {rows} x {cols} batch {batch} {dtype}", flush=True)
        assert torch.equal(ops.gemv_stage_forward(x, s_col, bits, None), ops.gemv_stage_forward(xa, sa, bits, None))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ranks", [(64,), (832, 288), (96, 40), (5, 3), (40, 700), (128, 64, 32), (33, 300, 7, 64)])
@pytest.mark.parametrize("batch", [1, 4, 18])
def test_sums_of_terms(dev, batch, ranks, dtype):
    # pairs of terms share a launch; odd numbers of terms, terms whose intermediates do not fit the scratch side by
    # side and more than two terms go through fp32 partial sums
    m, n = 1030, 768
    terms, ref = [], 0
    x = _cast(oracle.synth_x(batch, n, 5), dtype)
    for i, r in enumerate(ranks):
        vt, u, *scales = oracle.synth_term(m, n, r, 60 + i)
        si, sm, so = (_cast(a, dtype) for a in scales)
        if i == 1:
            sm = None
        ref = ref + oracle.layer_forward(x.double().numpy(), vt, u, si.double().numpy(), None if sm is None else sm.double().numpy(),
                                         so.double().numpy(), dtype=np.float64)
        pk = lambda w: packing.binary_packer(torch.from_numpy(w), "half2").to(dev)
        terms.append((si.to(dev), pk(vt), None if sm is None else sm.to(dev), pk(u), so.to(dev)))
    print(f"sum of terms {ranks} batch {batch} {dtype}", flush=True)
    y = ops.gemv_mixture_forward(x.to(dev), terms)
    torch.cuda.synchronize()
    _close_in_norm(y, ref, dtype, 3)
