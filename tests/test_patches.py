"""The patch partitions behind the tracer transport's kernels (host tables,
no GPU): the batched form's fused kernel (three rings) and trcadv12, and the
FP64 step's trcadv1 (two).  Every cell is in exactly one patch's core; a
patch's rings are exactly the cells at neighbour distance 1, 2 and 3 from its
core; the local neighbour table of all but the last ring points at the right
cells inside the tile (with each cell's edge count and its neighbours' edge
slots, and in the FP64 tables each core cell's pentagon neighbours); and the
sizes stay within the kernel's LDS tile (local indices fit in 8 bits)."""
import numpy as np
import pytest

from fimocn_subx_realtime_hera_apr2020_amd import fimhip, glvl
from helpers import golden_grid

# the kernel's LDS tile (ens_internal.h): core, rings 0-1, 0-2, 0-3
LIMITS = ((64, 112, 160, 208), (48, 84, 124, 124), (44, 80, 120, 120))
assert max(max(x) for x in LIMITS) <= 256


def _check(grid, form=0, core=0):
    cnt, ent = fimhip.patches(grid, form, core)
    CORE_MAX, R_MAX, LO_MAX, TILE_MAX = LIMITS[form]
    CORE_MAX = min(core, CORE_MAX) if core else CORE_MAX
    rings = 3 if form == 0 else 2
    prox = np.asarray(grid.prox, np.int64) - 1
    proxs = np.asarray(grid.proxs, np.int64) - 1
    nprox = np.asarray(grid.nprox)
    for c in np.where(nprox == 5)[0]:
        prox[c, 5] = prox[c, 4]
        proxs[c, 5] = proxs[c, 4]
    nip = grid.nip
    seen = np.zeros(nip, np.int64)
    off = 0
    for n0, n1, n2, n3 in cnt:
        ends = (0, n0, n1, n2, n3)
        assert 1 <= n0 <= CORE_MAX and n1 <= R_MAX and n2 <= LO_MAX and n3 <= TILE_MAX
        assert n0 <= n1 <= n2 <= n3
        cells = ent[off:off + n3, 0].astype(np.int64)
        assert cells.min() >= 0 and cells.max() < nip and len(set(cells.tolist())) == n3
        seen[cells[:n0]] += 1
        # rings by breadth-first distance from the core
        dist = {int(c): 0 for c in cells[:n0]}
        front = list(dist)
        assert rings == 3 or n3 == n2
        for r in range(1, rings + 1):
            nxt = sorted({int(x) for c in front for x in prox[c] if int(x) not in dist})
            for x in nxt:
                dist[x] = r
            front = nxt
        for r in range(1, rings + 1):
            ring = cells[ends[r]:ends[r + 1]].tolist()
            assert ring == sorted(x for x, d in dist.items() if d == r), (r, ring[:5])
        # local neighbour table of all but the last ring
        for i in range(ends[rings]):
            e4 = ent[off + i].astype(np.int64) & 0xFFFFFFFF
            loc = [(e4[1] >> 8 * e) & 0xFF for e in range(4)] + [(e4[2] >> 8 * e) & 0xFF for e in range(2)]
            assert (e4[2] >> 16) & 0xFF == nprox[cells[i]]
            assert [(e4[3] >> 4 * e) & 0xF for e in range(6)] == [int(x) for x in proxs[cells[i]]]
            assert max(loc) < n3
            assert [int(cells[l]) for l in loc] == [int(x) for x in prox[cells[i]]]
            if i < n1:
                assert max(loc) < n2          # ring-1 neighbours lie in rings 0-2
            if form == 2 and i < n0:
                assert [(e4[2] >> 24 + e) & 1 for e in range(6)] == [int(nprox[x] == 5) for x in prox[cells[i]]]
            if i < n0:
                assert max(loc) < n1          # core neighbours lie in rings 0-1
        off += n3
    assert off == len(ent)
    assert np.all(seen == 1)
    return cnt


@pytest.mark.parametrize("level", [1, 2, 3])
def test_patches_of_the_golden_grids(level):
    _check(golden_grid(level))


def test_patches_of_g6_and_a_concatenated_grid():
    g6 = fimhip.icos_grid(6)
    cnt = _check(g6)
    # compact patches: the three rings hold about twice the core's cells
    assert cnt[:, 3].sum() / cnt[:, 0].sum() < 3.2
    assert cnt[:, 0].mean() > 60
    _check(glvl.concat([golden_grid(2), golden_grid(3)]))


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("core", [1, 12, 17, 30, 0])
def test_two_ring_patches(form, core):
    """The default steps' partitions, at the smallest core the small grids get
    (12 cells), odd ones and the form's limit."""
    for level in (1, 2, 3):
        _check(golden_grid(level), form, core)
    _check(fimhip.icos_grid(4), form, core)
    _check(glvl.concat([golden_grid(2), golden_grid(3)]), form, core)


@pytest.mark.parametrize("form", [1, 2])
def test_two_ring_patches_of_larger_grids(form):
    _check(fimhip.icos_grid(5), form)
    cnt = _check(fimhip.icos_grid(6), form)
    # compact patches: the two rings hold about 1.5 times the core's cells
    assert cnt[:, 2].sum() / cnt[:, 0].sum() < 2.8
    assert cnt[:, 0].mean() > 40
