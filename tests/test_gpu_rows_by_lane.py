"""Backward kernels that give a lane a whole query, by rows of every width they take:
rows that end in another 64-byte line than they start in, ordered queries (through the
tables of lines), unordered ones (past them, two corners at a time) and tiles of both;
either side of the number of queries from which narrow rows are scattered that way and
of the one from which the cells' codes stand in LDS."""
import pytest
import torch

from helpers import assert_close_sums
from test_gpu_query import ATOL32, RTOL32, _eps

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
_NARROW, _LDS = 3 << 15, (1 << 19) + 1


def _operands(width, n, cells, seed):
    """Queries of 40 (5000) blocks with any tables, some corners in missing blocks: a third in
    order, a third in none, then stretches of 37 of either."""
    g = torch.Generator().manual_seed(seed)
    blocks = 40 if n < _LDS else 5000
    lut_g = torch.randint(0, blocks, (blocks, 8), generator=g)
    lut_g[:, 0] = torch.arange(blocks)
    lut_g[1, 5] = -1
    c2c, c2g = torch.randint(0, cells, (cells, 8), generator=g), torch.randint(0, 8, (cells, 8), generator=g)
    c2c[:, 0], c2g[:, 0] = torch.arange(cells), 0
    c2c[:-1, 1], c2g[:, 1] = torch.arange(1, cells), 0   # (the x neighbour is the next row)
    i = torch.arange(n)
    gi, ci = i * 5 // 997 % blocks, i // 3 % cells
    loose = (i >= n // 3) & ((i < 2 * n // 3) | (i // 37 % 2 == 0))
    gi = torch.where(loose, torch.randint(0, blocks, (n,), generator=g), gi)
    ci = torch.where(loose, torch.randint(0, cells, (n,), generator=g), ci)
    emb = torch.rand(blocks, cells, width, generator=g) - 0.5
    ops = (emb, torch.rand(n, 3, generator=g), gi, ci, torch.rand(n, generator=g) < 0.95, lut_g, c2c, c2g)
    rest = tuple(torch.rand(n, w, generator=g) - 0.5 for w in (width, 3, width))
    return ops, rest


@pytest.mark.parametrize("width,n,cells", [
    (width, n, 64) for width in (1, 2, 3, 5, 6, 7, 8, 12, 16) for n in (1, 65, 5003)]
    + [(width, n, 512) for width in (1, 2) for n in (_NARROW - 1, _NARROW)]
    + [(width, _LDS, 512) for width in (1, 2, 3, 6, 7, 8, 12, 16)] + [(5, _LDS, 577), (3, _LDS, 577)])
def test_every_gradient_against_the_oracle(gpu_ash, oracle, width, n, cells):
    ops, (z, u, z2) = _operands(width, n, cells, seed=width + n)
    dev = tuple(t.to(DEV) for t in ops)
    backend = gpu_ash.grid_query.backend
    dense = dict(eps=_eps(torch.float32), rtol=RTOL32, atol=ATOL32)
    per_query = dict(rtol=RTOL32, atol=ATOL32)
    sums = oracle.query_term_sums(u, z, *ops, 2, "smooth_step")
    ge_ref, go_ref = oracle.query_backward_forward(z, *ops, 2, "smooth_step")
    gz_ref, ge2_ref, _ = oracle.query_backward_backward(None, u, z, *ops, 2, "smooth_step")
    # either gradient and both
    for kinds in ((True, True), (True, False), (False, True)):
        ge, go = backend.query_backward_forward(z.to(DEV), *dev, 2, "smooth_step",
                                                need_embeddings=kinds[0], need_offsets=kinds[1])
        if kinds[0]:
            assert_close_sums(ge, ge_ref, sums["bf_embeddings"], what="grad_embeddings", **dense)
        if kinds[1]:
            assert torch.allclose(go.cpu(), go_ref, **per_query)
        gz, ge, _ = backend.query_backward_backward(None, u.to(DEV), z.to(DEV), *dev, 2, "smooth_step",
                                                    need_z=kinds[1], need_embeddings=kinds[0])
        if kinds[0]:
            assert_close_sums(ge, ge2_ref, sums["bb_embeddings"], what="second order", **dense)
        if kinds[1]:
            assert torch.allclose(gz.cpu(), gz_ref, **per_query)
    # both orders in one scatter
    both_ref = ge_ref + oracle.query_backward_backward(None, u, z2, *ops, 2, "smooth_step")[1]
    both = sums["bf_embeddings"] + oracle.query_term_sums(u, z2, *ops, 2, "smooth_step")["bb_embeddings"]
    for need_offsets in (True, False):
        ge, go = backend.host.query_backward_both(z.to(DEV), u.to(DEV), z2.to(DEV), list(dev), "smooth_step",
                                                  need_offsets, None)
        assert_close_sums(ge, both_ref, both, what="both orders", **dense)
        if need_offsets:
            assert torch.allclose(go.cpu(), go_ref, **per_query)


@pytest.mark.parametrize("width", [1, 2, 3, 4, 5, 7, 8, 12, 16])
@pytest.mark.parametrize("n", [5003, _NARROW - 1, _NARROW, _LDS])
def test_a_query_gets_the_same_whatever_else_is_asked_for(gpu_ash, width, n):
    """To the bit, whichever kernels the sizes and the gradients asked for choose."""
    ops, (z, u, z2) = _operands(width, n, 64, seed=width)
    dev = [t.to(DEV) for t in ops]
    z, u, z2 = z.to(DEV), u.to(DEV), z2.to(DEV)
    backend = gpu_ash.grid_query.backend
    alone = backend.query_backward_forward(z, *dev, 2, "smooth_step", need_embeddings=False, need_offsets=True)[1]
    for both in (backend.query_backward_forward(z, *dev, 2, "smooth_step")[1],
                 backend.host.query_backward_both(z, u, z2, dev, "smooth_step", True, None)[1]):
        assert torch.equal(alone, both)
    alone = backend.query_backward_backward(None, u, z, *dev, 2, "smooth_step", need_embeddings=False)[0]
    assert torch.equal(alone, backend.query_backward_backward(None, u, z, *dev, 2, "smooth_step")[0])
