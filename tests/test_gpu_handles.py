"""Lattice handles that change or are replaced while something else holds what it read from them."""
import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(bmx):
    c = bmx.tracking.Context(0)
    c.set_maps("fast")
    return c


def _same(a, b):
    for k in P.KEYS:
        bits = np.int64 if a[k].dtype == np.float64 else np.int32
        bad = np.nonzero(a[k].view(bits) != b[k].view(bits))[0]
        assert bad.size == 0, (k, bad.size, bad[:5], a[k][bad[:5]], b[k][bad[:5]])


def test_specialising_lattices_that_are_served(bmx, ctx):
    """Lattices specialised while a server tracks requests through them (in chunks of 2 turns, so that
    the server reads each lattice before, during and after): the results of each lattice alone, bit
    for bit (a ring without cavities and with all elements on operations)."""
    T, L = bmx.tracking, bmx.lattices
    arrs = [bmx.elements.to_array(v[:-1]) for v in L.ring1_variants(3, 3, n_cells=12)]
    beams = [P.random_beam(bmx, 300 + 100 * i, i) for i in range(6)]
    want = [T.track_beam_host(arrs[i % 3], b, 60) for i, b in enumerate(beams)]
    lats = [T.Lattice(ctx, a) for a in arrs]
    server = T.Server(ctx, 64 << 20, chunk_turns=2)
    print("served lattices", flush=True)
    ids = [server.submit(lats[i % 3], b, 60) for i, b in enumerate(beams)]
    for lat in lats:
        assert lat.specialize()
    late = [server.submit(lats[i % 3], b, 60) for i, b in enumerate(beams)]
    for i, (first, second) in enumerate(zip(ids, late)):
        _same(server.wait(first)[0], want[i])
        _same(server.wait(second)[0], want[i])
    server.close()
    for lat in lats:
        lat.close()
