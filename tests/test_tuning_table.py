"""The committed launch-shape decisions are ones that the pair pass looks up (no GPU)."""
import os

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llnl-spheral_amd", "tuning",
                     "mi355x_gfx950.txt")

# nodes up to which the pass gives a node several lanes and has one launch shape (lanes.hh)
SEVERAL_LANES = {(1, 0): 32768, (1, 1): 0, (2, 0): 49152, (2, 1): 98304}


def test_decisions_are_reachable():
    rows = [l.split() for l in open(TABLE) if l.strip() and not l.startswith("#")]
    assert rows
    for r in rows:
        dim, precision, size = int(r[1]), int(r[2]), int(r[4])
        assert 2 ** (size + 1) - 1 > SEVERAL_LANES[dim, precision], r
