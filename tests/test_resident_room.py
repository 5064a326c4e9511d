"""Which Krylov runs may be on the chip at once (host only).

A run waits for all of its blocks, so two runs admitted together must both get
all of theirs, however the dispatcher interleaves them.  The model here is the
worst case: the blocks of a launch go to the 8 XCDs in turn, and a block takes a
compute unit (CU) that none of the run's blocks is on for as long as there is
one without foreign blocks; a CU that holds blocks of one run takes none of
another.  A run alone may put up to its occupancy on a CU."""
import itertools

import numpy as np
import pytest

XCDS, CUS = 8, 256
TILES = sorted({1, 2, 7, 8, 9, 18, 45, 63, 64, 65, 95, 96, 97, 127, 128, 129, 153, 247, 248, 249, 255, 256, 257, 300, 318,
                384, 385, 512, 561, 768} | set(np.random.default_rng(5).integers(1, 768, 30).tolist()))


def _all_resident(tiles, first):
    """Whether every block of the runs finds a place: run ``first`` is
    dispatched whole before the others, so it spreads as far as it can."""
    per = CUS // XCDS
    for x in range(XCDS):
        free = per
        for k in [first] + [k for k in range(len(tiles)) if k != first]:
            blocks = len(range(x, tiles[k], XCDS))
            if blocks > free:
                return False
            free -= blocks
    return True


def _admitted(tiles, units):
    return sum(units(t) for t in tiles) <= CUS


def test_admitted_runs_are_resident_together():
    from pybella_amd import _abi
    lib = _abi.load()
    units = lambda t: lib.pb_resident_units(t, CUS)
    seen = 0
    for pair in itertools.combinations_with_replacement(TILES, 2):
        if _admitted(pair, units):
            seen += 1
            assert all(_all_resident(pair, f) for f in (0, 1)), pair
    for trio in itertools.combinations_with_replacement([t for t in TILES if t <= 130], 3):
        if _admitted(trio, units):
            seen += 1
            assert all(_all_resident(trio, f) for f in (0, 1, 2)), trio
    assert seen > 500
    assert not _admitted((300, 318), units) and _admitted((45, 153), units)


def test_the_model_tells_an_account_that_assumes_packed_blocks():
    packed = lambda t: -(-t // 2)   # two blocks per CU
    assert any(_admitted(p, packed) and not _all_resident(p, 0)
               for p in itertools.combinations_with_replacement(TILES, 2))


@pytest.mark.parametrize("tiles,cus,want", [(1, 256, 8), (8, 256, 8), (9, 256, 16), (249, 256, 256), (256, 256, 256),
                                            (768, 256, 256), (5, 32, 8), (40, 32, 32), (0, 256, -1), (4, 0, -1)])
def test_units(tiles, cus, want):
    from pybella_amd import _abi
    assert _abi.load().pb_resident_units(tiles, cus) == want
