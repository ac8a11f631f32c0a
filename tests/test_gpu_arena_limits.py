"""Counts in arenas of growing size: too small for either order of the
symmetry conditions, large enough for conditions by vertex id only, and for
those by degree.  A match gives its count or FSIG_ENOMEM, says nothing of a
first attempt that did not fit, and leaves the context as it was; with and
without event timing."""
import numpy as np
import pytest

import fsig_amd as F

pytestmark = pytest.mark.gpu

BOWTIE = F.Query(5, np.zeros(5, np.int32), [(0, 1), (1, 2), (0, 2), (2, 3), (3, 4), (2, 4)])
EDGE = F.Query(2, np.zeros(2, np.int32), [(0, 1)])
FILTER = F.KERNEL_FAMILIES.index("filter")


@pytest.mark.parametrize("profiling", [False, True])
def test_counts_in_small_arenas(profiling):
    g = F.HostGraph.rmat(13, 60000, seed=3)
    big = F.Context(0, 1 << 30)
    dg = big.upload(g)
    want = F.match(dg, BOWTIE).count
    want_edge = F.match(dg, EDGE).count
    dg.free()
    big.close()
    seen = set()
    for kib in range(512, 12288, 192):
        ctx = F.Context(0, kib << 10)
        dg = ctx.upload(g)
        ctx.set_profiling(profiling)
        try:
            assert F.match(dg, BOWTIE).count == want, kib
            assert ctx._L.fsig_last_error(ctx._h) == b"", kib
            tries = ctx.kernel_stats(FILTER)["launches"]
            assert not profiling or ctx.kernel_stats(FILTER)["ms"] > 0
        except F.FsigError as e:
            assert e.code == F.FSIG_ENOMEM and "arena exhausted" in str(e), (kib, e)
            tries = 0
        seen.add(tries)
        try:  # the next match, of a query that needs less
            assert F.match(dg, EDGE).count == want_edge, kib
        except F.FsigError as e:
            assert e.code == F.FSIG_ENOMEM and tries == 0, (kib, e)
        dg.free()
        ctx.close()
        if tries == 1:
            break
    assert seen == {0, 1, 2}  # neither order fits; by degree; by id after the other did not
