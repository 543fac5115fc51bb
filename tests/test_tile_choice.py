"""The choice of prefill tiles, on the host."""
import ctypes

import pytest

from nanoquant_amd import _lib, ops

ALONE, GROUP, ANY, SUM = range(4)


def tile(use, tokens, k, rows, scaled=False, nxt=None):
    """(tokens, rows) of the tile that a launch takes, None where it is refused."""
    ints = lambda a: None if a is None else (ctypes.c_int * len(a))(*a)
    size = _lib.lib().nq_gemm_tile_size(use, len(k), tokens, ints(k), ints(rows), int(scaled), ints(nxt))
    return (size >> 16, size & 0xFFFF) if size else None


def sum_route(tokens, weights):
    """Tile of the launch that sums the terms (n, r, m) of every weight, and whether gemm_group_sum_forward makes it."""
    order = sorted(range(len(weights)), key=lambda w: -len(weights[w]))
    flat = [(w, t) for t in range(len(weights[order[0]])) for w in order if t < len(weights[w])]      # as the call lists them
    nxt = [flat.index((w, t + 1)) if (w, t + 1) in flat else -1 for w, t in flat]
    sizes = [weights[w][t] for w, t in flat]
    arr = (ops.NqGemmTerm * len(flat))(*[ops.NqGemmTerm(4096, 4096, 4096, 4096, None, None, None, 4096 * (i + 1), 16 * (i + 1), *s)
                                         for i, s in enumerate(sizes)])      # addresses that nobody reads
    pays = _lib.lib().nq_gemm_sum_pays(arr, (ctypes.c_int * len(flat))(*nxt), len(flat), tokens)
    return tile(SUM, tokens, [r for _, r, _ in sizes], [m for _, _, m in sizes], nxt=nxt), pays == 1


def test_sizes_that_are_refused():
    assert tile(ALONE, 5, [256], [32]) == (32, 32)
    for use, tokens, k, rows, nxt in [(ALONE, 0, [256], [32], None), (ALONE, 5, [0], [32], None), (ALONE, 5, [256], [0], None),
                                      (ALONE, 5, [300], [32], None), (ALONE, 5, [256], [33], None), (4, 5, [256], [32], None),
                                      (SUM, 5, [256], [32], None), (ANY, 5, [256], [32], [-1]), (SUM, 5, [256], [32], [0]),
                                      (SUM, 5, [256], [32], [1]), (SUM, 5, [256, 256], [32, 64], [1, -1])]:
        assert tile(use, tokens, k, rows, nxt=nxt) is None


# {q, k, v} and {gate, up} in two terms each: 64 x 256 tiles hold the sums twice, two workgroups to a compute unit.  us of both
# stages on 64 x 128 / 64 x 256
@pytest.mark.parametrize("tokens,k,rows", [
    (333, [1536, 768, 768, 512, 256, 256], [4096, 1024, 1024]),      # 33.6 / 37.5
    (512, [1536, 768, 768, 512, 256, 256], [4096, 1024, 1024]),      # 38.4 / 41.7
    (160, [2048, 2048, 768, 768], [11008, 11008]),                   # 41.0 / 44.2
])
def test_sums_are_priced_by_the_workgroups_that_fit(tokens, k, rows):
    n = len(rows)
    assert tile(SUM, tokens, k, rows * 2, nxt=[n + i for i in range(n)] + [-1] * n) == (64, 128)
