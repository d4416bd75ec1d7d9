"""The page form of the strand expansion (256 consecutive vertices of every
instance a workgroup): one-line settings at any size, more lines above the
output size where it takes over, pages that start inside a patch, a partial
last page, a single triangle.  The oracle's operations in the oracle's order:
bit for bit."""
import numpy as np
import pytest

import barbu_amd as ba
from oracle import ftl_oracle as orc
from tests.helpers import assert_bitexact
from tests.test_expand import scene

pytestmark = pytest.mark.gpu


def check(ctx, S, N, T, ninst, nlines, nsub):
    print("expand pages S=%d N=%d T=%d %d x %d x %d" % (S, N, T, ninst, nlines, nsub), flush=True)
    pos, tan, tris, rnd = scene(S, N, T, R=4096, seed=S + nsub)
    g = ba.Groom(ctx, pos)
    e = ba.Expand(ctx, S, N, tris, tan, rnd)
    got = e.run_groom(g, ba.expand_params(ninst, nlines, nsub, 1.1))
    want = orc.expand_f32(pos, tan, tris, rnd, ninst, nlines, nsub, 1.1)
    assert_bitexact(got, want, "expansion")
    e.close()
    g.close()


@pytest.mark.parametrize("T", [1, 3, 257])
@pytest.mark.parametrize("ninst,nsub", [(1, 6), (2, 7), (1, 13), (2, 10), (1, 33), (2, 64), (1, 63)])
def test_one_line(ctx, T, ninst, nsub):
    check(ctx, 60, 5, T, ninst, 1, nsub)


@pytest.mark.parametrize("ninst,nlines,nsub", [(3, 2, 7), (3, 3, 10), (2, 5, 5), (4, 1, 14)])
def test_large_outputs(ctx, ninst, nlines, nsub):
    per = 2 * ninst * nlines * nsub * 15
    check(ctx, 2000, 16, (384 << 20) // (16 * per) + 3, ninst, nlines, nsub)


@pytest.mark.parametrize("above", [-1, 2])
@pytest.mark.parametrize("mb,ninst,nlines,nsub", [(128, 2, 1, 13), (224, 1, 1, 15), (224, 2, 1, 8), (224, 1, 3, 16),
                                                  (256, 2, 3, 6), (144, 3, 2, 9), (256, 4, 3, 8), (400, 3, 2, 7), (384, 3, 2, 16)])
def test_cache_lines(ctx, mb, ninst, nlines, nsub, above):
    """On both sides of the output sizes at which a form changes how its stores
    use the caches: pages, batches and single vertices, with ends that fill no
    page, batch or workgroup."""
    per = 2 * ninst * nlines * nsub * 15
    check(ctx, 2000, 16, (mb << 20) // (16 * per) + above, ninst, nlines, nsub)


@pytest.mark.parametrize("T", [1, 2, 5, 13, 129])
@pytest.mark.parametrize("ninst,nlines,nsub", [(1, 1, 1), (3, 2, 5), (2, 5, 2), (1, 1, 8), (3, 2, 16), (5, 2, 12), (8, 4, 64)])
def test_ends(ctx, T, ninst, nlines, nsub):
    """The last batch and the last workgroup hold fewer patches."""
    check(ctx, 40, 4, T, ninst, nlines, nsub)


@pytest.mark.parametrize("above", [-1, 2])
@pytest.mark.parametrize("mb,ninst,nlines,nsub", [(256, 3, 1, 8), (256, 5, 1, 8), (384, 2, 2, 12), (384, 4, 2, 8), (384, 1, 4, 16),
                                                  (224, 2, 1, 26), (256, 4, 4, 8), (400, 4, 4, 8)])
def test_store_lines(ctx, mb, ninst, nlines, nsub, above):
    """The same for batches of few and of many vertices a patch, one-line pages
    of many, and the per-vertex form's plain stores."""
    per = 2 * ninst * nlines * nsub * 15
    check(ctx, 2000, 16, (mb << 20) // (16 * per) + above, ninst, nlines, nsub)
