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


def test_plain_turns_of_replaced_lattices(bmx, ctx):
    """The plain path keeps a captured turn from call to call: lattices of equal length and different
    maps, each made after the one before was destroyed (their tables may come back at the same
    addresses), and radiation settings changed between calls, each as on the persistent kernel
    (losses identical, survivors within the per-element bar, 1e-12, for each element passed)."""
    E, T = bmx.elements, bmx.tracking
    p0c, et = bmx.lattices.reference()
    mk = lambda key, **kw: E.make_element(key, p0c, et, **kw, x_limit=0.02, y_limit=0.02)  # noqa: E731
    d, b = mk(E.DRIFT, l=0.5), mk(E.SBEND, l=1.0, g=0.02)
    q = mk(E.QUADRUPOLE, l=0.3, k1=0.2)
    q2 = mk(E.QUADRUPOLE, l=0.3, k1=-0.2, b_pole={2: 2.0}, num_steps=2)
    off = mk(E.QUADRUPOLE, l=0.3, k1=-0.2, x_offset=1e-4, tilt=0.1)
    beam = P.random_beam(bmx, 300, 6, scale=10.0, pz_sigma=1e-3)
    gb = T.Beam.from_host(ctx, beam)
    for again in range(2):
        for name, cell, rad in (("plain", [d, q, d, b], False), ("stepped", [d, q2, d, b], False),
                                ("radiating", [d, q, d, b], True), ("offset", [d, off, d, b], False),
                                ("stepped radiating", [d, q2, d, b], True), ("drifts", [d] * 4, False)):
            arr = E.to_array(cell * 6)
            maps = T.rad_maps(len(arr)) if rad else None
            if rad:
                maps["damp_dmat"][3::4, :, 5, 5] = -1e-4
                maps["stoc_mat"][3::4, :, 5, 5] = 1e-5
            lat = T.Lattice(ctx, arr, rad_maps=maps, rad=T.rad_config(True, True, seed=3) if rad else None)
            for seed in ((3, 4) if rad else (0,)):
                if seed == 4:
                    lat.set_radiation(T.rad_config(True, True, seed=seed))
                print(f"plain turns {name} pass {again} seed {seed}", flush=True)
                outs = []
                for track in (T.track_beam_plain, T.track_beam):
                    gb.upload(beam)
                    track(ctx, lat, gb, 2, 0)
                    ctx.synchronize()
                    outs.append(gb.download())
                assert P.loss_mismatch(*outs).size == 0, name
                alive = outs[1]["state"] == 1
                assert alive.sum() > 50
                assert P.rel_err(outs[0], outs[1], alive) <= 1e-12 * 2 * len(arr), name
            lat.close()
    gb.close()


def test_served_requests_keep_their_radiation_settings(bmx, ctx):
    """A lattice's radiation settings changed while a request through it waits or runs (chunks of 2
    turns): the request keeps those it was submitted with, the next one has the new ones; each
    bit-identical to its beam alone with them."""
    E, T = bmx.elements, bmx.tracking
    arr = E.to_array(bmx.lattices.ring1(n_cells=6))
    maps = T.rad_maps(len(arr))
    bends = np.nonzero(arr["key"] == E.SBEND)[0]
    maps["damp_dmat"][bends, :, 5, 5] = -1e-4
    maps["stoc_mat"][bends, :, 5, 5] = 1e-5
    cfgs = [T.rad_config(True, True, seed=1), T.rad_config(True, True, scale=2.0, seed=2)]
    beam = P.random_beam(bmx, 400, 3)
    lat = T.Lattice(ctx, arr, rad_maps=maps, rad=cfgs[0])
    server = T.Server(ctx, 64 << 20, chunk_turns=2)
    print("served radiation settings", flush=True)
    first = server.submit(lat, beam, 60)
    lat.set_radiation(cfgs[1])
    second = server.submit(lat, beam, 60)
    outs = [server.wait(r)[0] for r in (first, second)]
    server.close()
    lat.close()
    for out, cfg in zip(outs, cfgs):
        _same(out, T.track_beam_host(arr, beam, 60, rad_maps=maps, rad=cfg))
