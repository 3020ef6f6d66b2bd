"""Cell-specialised kernels on lattices whose cells differ in their strengths and apertures, and on
cells of every length the kernels' value lines treat differently: against the generic kernel."""
import numpy as np
import pytest

import parity as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(bmx):
    c = bmx.tracking.Context(0)
    c.set_maps("fast")
    return c


def _track(bmx, ctx, arr, beam, special, n_turns=2):
    T = bmx.tracking
    lat = T.Lattice(ctx, arr)
    if special:
        assert lat.specialize()
    b = T.Beam.from_host(ctx, beam)
    T.track_beam(ctx, lat, b, n_turns, 0)
    ctx.synchronize()
    out = b.download()
    b.close()
    lat.close()
    return out


def _same(a, b):
    for k in P.KEYS:
        bits = np.int64 if a[k].dtype == np.float64 else np.int32
        bad = np.nonzero(a[k].view(bits) != b[k].view(bits))[0]
        assert bad.size == 0, (k, bad.size, bad[:5], a[k][bad[:5]], b[k][bad[:5]])


# Cells by the kinds of their elements, and the values they have in the cell kernels' lines of 8: an
# aperture (2, here the same in every cell) and 1 for a drift, 2 for a kicker, 3 for a quadrupole or a
# sextupole, 6 for a bend.
CELLS = {
    "q": 5, "b": 8, "dq": 6, "dk": 5, "kq": 7, "qs": 8, "ddq": 7,  # one line
    "qds": 9, "dqdb": 15, "qsbdd": 16, "dqsdbdqsb": 33,            # several
    "dqkdsqbdqskdqsbdqdb": 70,                                     # several runs of operations
}


def _cells(bmx, kinds, seed, apertures=False):
    """24 cells (8 long ones) of the given kinds, each element with strengths of its own (the sign of
    k1 changes from quadrupole to quadrupole and from cell to cell) and all of them on operations;
    apertures: half-axes that change from cell to cell as well."""
    E = bmx.elements
    p0c, et = bmx.lattices.reference()
    rng = np.random.default_rng(seed)
    out = []
    for c in range(24 if len(kinds) < 10 else 8):
        s = rng.uniform(0.5, 1.0, len(kinds))
        for i, (kind, w) in enumerate(zip(kinds, s)):
            sign = (-1) ** (c + kinds[:i].count("q"))
            ap = dict(x_limit=0.02 * (w if apertures else 1.0), y_limit=0.02, aperture_type=E.APERTURE_ELLIPTICAL)
            mk = lambda key, **kw: E.make_element(key, p0c, et, **kw, **ap)  # noqa: E731, B023
            out.append({
                "d": lambda: mk(E.DRIFT, l=0.4 * w),
                "q": lambda: mk(E.QUADRUPOLE, l=0.3, k1=sign * 0.5 * w),
                "s": lambda: mk(E.SEXTUPOLE, l=0.2, k2=sign * 2.0 * w, num_steps=1),
                "k": lambda: mk(E.KICKER, hkick=1e-6 * w, vkick=-1e-6 * w),
                "b": lambda: mk(E.SBEND, l=1.0, g=0.016 + 0.005 * w),
            }[kind]())
    return out


@pytest.mark.parametrize("kinds, ends", [(k, False) for k in CELLS] +
                         [(k, True) for k in ("q", "dq", "qds", "dqkdsqbdqskdqsbdqdb")])
def test_cells_of_their_own_strengths(bmx, ctx, kinds, ends):
    """A ring of cells with strengths of their own, alone or with a head and a tail of other
    elements: the cell kernel and the generic one give the same bits, with lost particles among
    the others and without."""
    E = bmx.elements
    p0c, et = bmx.lattices.reference()
    eles = _cells(bmx, kinds, 11)
    if ends:
        mk = lambda **kw: E.make_element(E.QUADRUPOLE, p0c, et, l=0.2, tilt=0.3, **kw)  # noqa: E731
        eles = [mk(k1=0.02 * (-1) ** i) for i in range(len(kinds))] + eles + [mk(k1=-0.02)]
    arr = E.to_array(eles)
    for scale in (1.0, 40.0):
        beam = P.random_beam(bmx, 1000, 3, scale=scale, pz_sigma=1e-3)
        print(f"cells {kinds} ends {ends} scale {scale}", flush=True)
        want = _track(bmx, ctx, arr, beam, False)
        assert (want["state"] == 1).sum() > 50
        if scale > 1 and "q" in kinds:
            assert (want["state"] != 1).sum() > 0
        _same(_track(bmx, ctx, arr, beam, True), want)


@pytest.mark.parametrize("kinds", ["q", "dq", "dqdb", "dqkdsqbdqskdqsbdqdb"])
def test_apertures_that_change_from_cell_to_cell(bmx, ctx, kinds):
    arr = bmx.elements.to_array(_cells(bmx, kinds, 12, apertures=True))
    beam = P.random_beam(bmx, 1000, 4, scale=25.0, pz_sigma=1e-3)
    print(f"cell apertures {kinds}", flush=True)
    _same(_track(bmx, ctx, arr, beam, True), _track(bmx, ctx, arr, beam, False))


@pytest.mark.parametrize("general_first", [False, True])
def test_radiating_lattices_of_the_same_cells(bmx, ctx, general_first):
    """Two radiating lattices of the same cells and length, the last element a plain bend in one and a
    bend with a sextupole part in the other, specialised one after the other: each as on the
    generic kernel (losses identical, survivors within the per-element bar, 1e-12, for each element
    passed: the general maps are contracted by the compiler for each kernel)."""
    E, T = bmx.elements, bmx.tracking
    p0c, et = bmx.lattices.reference()
    mk = lambda key, **kw: E.make_element(key, p0c, et, **kw, x_limit=0.02, y_limit=0.02)  # noqa: E731
    cells = 9 + general_first  # kernels of its own for each order
    cell = [mk(E.DRIFT, l=0.5), mk(E.SBEND, l=1.0, g=0.02), mk(E.QUADRUPOLE, l=0.3, k1=0.05)]
    ends = {False: mk(E.SBEND, l=1.0, g=0.02), True: mk(E.SBEND, l=1.0, g=0.02, b_pole={2: 20.0}, num_steps=2)}
    beam = P.random_beam(bmx, 500, 8, scale=3.0, pz_sigma=1e-3)
    held = []
    for general in (general_first, not general_first):
        arr = E.to_array(cell * cells + [ends[general]])
        maps = T.rad_maps(len(arr))
        for i in np.nonzero(arr["key"] == E.SBEND)[0]:
            maps["damp_dmat"][i, :, 5, 5] = -1e-5
            maps["stoc_mat"][i, :, 5, 5] = 1e-6
        outs = []
        for special in (False, True):
            lat = T.Lattice(ctx, arr, rad_maps=maps, rad=T.rad_config(True, True, seed=7))
            held.append(lat)
            if special:
                assert lat.specialize()
            b = T.Beam.from_host(ctx, beam)
            print(f"radiating lattices, general {general}, special {special}", flush=True)
            T.track_beam(ctx, lat, b, 2, 0)
            ctx.synchronize()
            outs.append(b.download())
            b.close()
        assert P.loss_mismatch(outs[1], outs[0]).size == 0, general
        alive = outs[0]["state"] == 1
        assert alive.sum() > 50
        assert P.rel_err(outs[1], outs[0], alive) <= 1e-12 * 2 * len(arr), general
    for lat in held:
        lat.close()


def _general(bmx, kind):
    E = bmx.elements
    p0c, et = bmx.lattices.reference()
    mk = lambda key, **kw: E.make_element(key, p0c, et, **kw, x_limit=0.02, y_limit=0.02)  # noqa: E731
    return {
        "octupole": lambda w: mk(E.OCTUPOLE, l=0.2, k3=50.0 * w),
        "long bend": lambda w: mk(E.SBEND, l=2.0, g=0.06 + 0.01 * w),
        "pitch": lambda w: mk(E.QUADRUPOLE, l=0.3, k1=0.03 * w, x_pitch=1e-4),
        "stepped": lambda w: mk(E.QUADRUPOLE, l=0.3, k1=0.03 * w, b_pole={2: 1.0}, num_steps=2),
        "general bend": lambda w: mk(E.SBEND, l=1.0, g=0.02, e1=0.02 * w, k1=1e-3, b_pole={2: 0.1}, num_steps=2),
        "multipole": lambda w: mk(E.MULTIPOLE, knl={2: 1.0 * w, 3: 5.0}),
        "cavity": lambda w: mk(E.RFCAVITY, l=0.5, voltage=1e6 * w, rf_frequency=500e6),
    }[kind]


@pytest.mark.parametrize("kind", ["octupole", "long bend", "pitch", "stepped", "general bend", "multipole", "cavity"])
def test_cells_with_elements_of_the_general_maps(bmx, ctx, kind):
    """Cells of operations with elements of the general maps among them, first, last and next to each
    other, of strengths of their own: losses as on the generic kernel, survivors within the
    per-element bar, 1e-12, for each element passed (the general maps are contracted by the compiler
    for each kernel). A beam that is partly lost, and one on and near the zero orbit."""
    E, L = bmx.elements, bmx.lattices
    p0c, et = L.reference()
    mk = lambda key, **kw: E.make_element(key, p0c, et, **kw, x_limit=0.02, y_limit=0.02)  # noqa: E731
    rng = np.random.default_rng(5)
    general = _general(bmx, kind)
    eles = []
    for c in range(10):
        a, b, w = rng.uniform(0.5, 1.0, 3)
        eles += [general(w), mk(E.DRIFT, l=0.4 * a), mk(E.QUADRUPOLE, l=0.3, k1=0.3 * a), general(a), general(b),
                 mk(E.SBEND, l=1.0, g=0.02), mk(E.QUADRUPOLE, l=0.3, k1=-0.3 * b), general(b)]
    arr = E.to_array(eles + [mk(E.DRIFT, l=0.1)])
    near = P.random_beam(bmx, 200, 2, scale=1e-3)
    for k in P.COORDS:
        near[k][:20] = 0
    near["pz"][:100] = 0
    near["beta"] = L.init_beta(near["pz"], p0c, et)
    for beam in (P.random_beam(bmx, 500, 2, scale=10.0, pz_sigma=5e-4), near):
        print(f"general cells {kind}", flush=True)
        want = _track(bmx, ctx, arr, beam, False)
        got = _track(bmx, ctx, arr, beam, True)
        assert P.loss_mismatch(got, want).size == 0
        alive = want["state"] == 1
        assert alive.sum() > 10
        assert P.rel_err(got, want, alive) <= 1e-12 * 2 * len(arr)


def test_cells_whose_elements_are_of_different_kinds_of_operation(bmx, ctx):
    """A cell position that is on the short series of the quadrupole in some cells and on the long one
    in others: the same bits as the generic kernel, which takes each element by its own."""
    E = bmx.elements
    p0c, et = bmx.lattices.reference()
    mk = lambda key, **kw: E.make_element(key, p0c, et, **kw, x_limit=0.02, y_limit=0.02)  # noqa: E731
    k1 = [0.6, -0.62, 0.61, -0.6] * 3
    eles = [e for c, k in enumerate(k1) for e in
            (mk(E.DRIFT, l=0.4), mk(E.QUADRUPOLE, l=0.3, k1=k), mk(E.DRIFT, l=0.2 + 0.01 * c))]
    print("cells of different operations", flush=True)
    arr = E.to_array(eles)
    beam = P.random_beam(bmx, 500, 2, scale=10.0)
    _same(_track(bmx, ctx, arr, beam, True), _track(bmx, ctx, arr, beam, False))
