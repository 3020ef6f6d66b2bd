"""Single-launch spans and the packing of live particles: the same bits as the chunked way."""
from __future__ import annotations

import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(bmx):
    c = bmx.tracking.Context(0)
    c.set_maps("fast")
    return c


def _lattice(bmx, ctx, kind):
    L, E, T = bmx.lattices, bmx.elements, bmx.tracking
    eles = list(L.ring1(n_cells=4))
    if kind == "stepped":  # a sextupole component makes a quadrupole a stepped one
        p0c, et = L.reference()
        eles[4:4] = [E.make_element(E.QUADRUPOLE, p0c, et, l=0.1, k1=0.1, b_pole={2: 5.0}, num_steps=2)]
    arr = E.to_array(eles)
    if kind != "radiation":
        return T.Lattice(ctx, arr), len(arr)
    maps = T.rad_maps(len(arr))
    for i in np.nonzero(arr["key"] == E.SBEND)[0]:
        for k in range(2):
            maps[i, k]["damp_dmat"][5, 5] = -1e-5
            maps[i, k]["stoc_mat"][5, 5] = 1e-6
    return T.Lattice(ctx, arr, rad_maps=maps, rad=T.rad_config(True, True, seed=7)), len(arr)


def _beam(bmx, n, seed):
    b = P.random_beam(bmx, n, seed, scale=20.0)
    dead = np.random.default_rng(seed).random(n) < 0.3
    b["state"][dead] = 4
    b["loss_ele"][dead] = 3
    return b


def _same(a, b):
    for k in P.KEYS:
        assert np.array_equal(a[k].view(np.int64) if a[k].dtype == np.float64 else a[k],
                              b[k].view(np.int64) if b[k].dtype == np.float64 else b[k]), k


@pytest.mark.parametrize("maps", ["fast", "reference"])
@pytest.mark.parametrize("kind", ["plain", "stepped", "radiation"])
def test_spans_in_one_launch(bmx, ctx, kind, maps):
    """Spans of a beam that fits on the card at once, against the same spans on a grid of one
    workgroup, whose four waves no beam of more than 256 particles fits: from and to elements
    inside, round the end, a whole turn from inside, and several turns (one chunk, and more).
    Bit for bit with the fast maps, whose operations fix every rounding; the reference maps and the stepped
    maps are contracted by the compiler for each kernel, so there losses are identical and survivors within the per-element
    bar, 1e-12, for each element passed."""
    T = bmx.tracking
    ctx.set_maps(maps)
    lat, n_ele = _lattice(bmx, ctx, kind)
    try:
        for n in (257, 1000):
            beam = _beam(bmx, n, n)
            for first, last, turns in ((3, 4, 1), (0, 17, 1), (11, n_ele - 2, 1), (n_ele - 5, 6, 1), (7, 7, 1),
                                       (9, None, 1), (9, None, 5), (9, None, 7)):
                print(f"span {kind} {maps} n={n} {first}..{last} turns {turns}", flush=True)
                outs = []
                for grid in (0, 1):
                    ctx.set_run(5, grid, 0)
                    b = T.Beam.from_host(ctx, beam)
                    if last is None:
                        T.track_beam_from(ctx, lat, b, first, turns, 2)
                    else:
                        T.track_bunch(ctx, lat, b, first, last, 2)
                    ctx.synchronize()
                    outs.append((b.download(), ctx.take_work()))
                    b.close()
                if maps == "fast" and kind != "stepped":
                    _same(outs[0][0], outs[1][0])
                else:
                    a, b = outs[0][0], outs[1][0]
                    assert P.loss_mismatch(a, b).size == 0
                    passed = (last - first) % n_ele if last not in (None, first) else n_ele
                    assert P.rel_err(a, b, b["state"] == 1) <= 1e-12 * passed * turns
                assert outs[0][1] == outs[1][1]
    finally:
        ctx.set_run(5, 0, 0)
        ctx.set_maps("fast")
        lat.close()


def test_packing_of_many_groups(bmx, ctx):
    """A batch of more tiles than the packing kernel has waves (several tiles per wave, groups that
    begin and end inside a wave's share, particles dead on arrival): each group as by itself."""
    E, L, T = bmx.elements, bmx.lattices, bmx.tracking
    lat = T.Lattice(ctx, E.to_array(L.ring1(n_cells=2)))
    rng = np.random.default_rng(5)
    counts = np.concatenate([[1, 63, 64, 65, 0, 511, 513], rng.integers(1, 16000, 60)])
    assert ((counts + 63) // 64).sum() > 2 * 2048
    first = np.concatenate([[0], np.cumsum(counts)[:-1]])
    beam = _beam(bmx, int(counts.sum()), 31)
    print("packing", int(counts.sum()), flush=True)
    b = T.Beam.from_host(ctx, beam)
    batch = T.Batch(ctx, [(lat, b, int(f), int(c)) for f, c in zip(first, counts)])
    batch.track(2)
    ctx.synchronize()
    got = b.download()
    batch.close()
    b.close()
    for f, c in zip(first[:12], counts[:12]):
        if c == 0:
            continue
        one = T.Beam.from_host(ctx, {k: v[f:f + c].copy() for k, v in beam.items()})
        T.track_beam(ctx, lat, one, 2)
        ctx.synchronize()
        _same({k: v[f:f + c].copy() for k, v in got.items()}, one.download())
        one.close()
    lat.close()
