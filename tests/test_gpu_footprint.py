"""pg_plan_footprint counts every buffer per entry that a forward pass holds."""
import numpy as np
import pytest

import subgraph_amd as sg


def _ring(n, h):
    """Vertices joined to the h next on a ring: 2 h neighbours each."""
    v = np.repeat(np.arange(n, dtype=np.int32), h)
    return sg.csc_from_edges(n, v, ((v + np.tile(np.arange(1, h + 1), n)) % n).astype(np.int32))


@pytest.mark.gpu
def test_device_bytes_per_entry():
    """Between rings of 4 and of 16 neighbours only the entries and the tiles
    change.  An entry: 4 bytes of neighbour, 4 of caller's entry, 1 of colour, 1 of
    place in its tile.  Tiles of 16 bytes: of 64 and 16 vertices (256 entries) and
    of 256 and 64 (1,024 entries, at most 256 vertices)."""
    n = 4096
    bytes_of = {}
    for h in (2, 8):
        ctx = sg.Context(0)
        ctx.upload_graph(*_ring(n, h))
        bytes_of[h] = ctx.footprint(ctx.plan(3, [(0, 1), (1, 2)]), 1)["device_bytes"]
    tiles = (n // 16 - n // 64) + (n // 64 - n // 256)
    assert bytes_of[8] - bytes_of[2] == 10 * 2 * (8 - 2) * n + 16 * tiles
