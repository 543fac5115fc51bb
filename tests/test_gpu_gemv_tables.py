"""Group decode launches by the number of linears: the kernels take tables of one, three and eight entries, and a linear gets the
same bits whichever table it sits in and wherever in it."""
import pytest
import torch

from nanoquant_amd import ops

pytestmark = pytest.mark.gpu


def _linear(dev, gen, m, n, r, dtype):
    words = lambda rows, cols: torch.randint(-2 ** 31, 2 ** 31 - 1, (rows, (cols + 31) // 32), dtype=torch.int32, device=dev, generator=gen)
    scale = lambda k: (torch.rand(k, device=dev, generator=gen) * 0.02 + 1e-3).to(dtype)
    return scale(n), words(r, n), scale(r), words(m, r), scale(m)


@pytest.mark.parametrize("count", [1, 2, 3, 4, 8, 9])
@pytest.mark.parametrize("rows", [1, 3, 16])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_bits_do_not_depend_on_the_table(dev, count, rows, dtype):
    gen = torch.Generator(device=dev)
    gen.manual_seed(count)
    # rows of 16 left over, ranks that are no multiple of 8, one linear much taller than the others
    sizes = [(48 + 40 * i if i != 1 else 4112, 512 + 64 * (i % 3), 96 + 31 * i) for i in range(count)]
    lins = [_linear(dev, gen, m, n, r, dtype) for m, n, r in sizes]
    xs = [torch.randn(rows, n, device=dev, generator=gen).to(dtype) for _, n, _ in sizes]
    print(f"table {count} linears {rows} rows {dtype}", flush=True)
    together = ops.gemv_group_forward(xs, lins)
    alone = [torch.ops.binary_kernels.nanoquant_dyn_forward(x, *lin) for x, lin in zip(xs, lins)]
    torch.cuda.synchronize()
    for a, y, (m, _, _) in zip(alone, together, sizes):
        assert y.shape == (rows, m) and torch.equal(a, y)
