"""Elements on their straight-line operations (csrc/bmx_fast.hpp): against the CPU restatement at
the limits of the operations' tests, and the same bits from every kernel that tracks them."""
import numpy as np
import pytest

import parity as P
import rad_fixtures as R

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx(bmx):
    c = bmx.tracking.Context(0)
    c.set_maps("fast")
    return c


def _apertures(bmx):
    E = bmx.elements
    return {
        "none": {},
        "ellipse": dict(x_limit=0.01, y_limit=0.006, aperture_type=E.APERTURE_ELLIPTICAL),
        "rectangle": dict(x_limit=0.01, y_limit=0.006, aperture_type=E.APERTURE_RECTANGULAR),
        # not about the axis: the general maps
        "off_axis": dict(x1_limit=0.01, x2_limit=0.02, y1_limit=0.005, y2_limit=0.006,
                         aperture_type=E.APERTURE_RECTANGULAR),
    }


def _elements(bmx, **ap):
    """Elements on both sides of each limit of the operations: the quadrupole's two series and the
    general map beyond them (k1 L^2 0.055 and 0.7), sextupoles of one and several steps, thin and
    thick kickers, bends (a weak one is the general maps'), gradient bends, offset and tilted
    magnets (a pitch is the general maps'), dipole kicks in quadrupoles."""
    E = bmx.elements
    p0c, et = bmx.lattices.reference()
    mk = lambda key, **kw: E.make_element(key, p0c, et, **kw, **ap)  # noqa: E731
    off = dict(x_offset=3e-4, y_offset=-2e-4, tilt=0.01)
    return {
        "drift": mk(E.DRIFT, l=1.3),
        "marker": mk(E.MARKER),
        "quad_weak": mk(E.QUADRUPOLE, l=0.3, k1=0.61),
        "quad_mid": mk(E.QUADRUPOLE, l=0.3, k1=-0.612),
        "quad_strong": mk(E.QUADRUPOLE, l=1.0, k1=0.69),
        "quad_general": mk(E.QUADRUPOLE, l=1.0, k1=0.71),
        "sext_1": mk(E.SEXTUPOLE, l=0.2, k2=20.0, num_steps=1),
        "sext_3": mk(E.SEXTUPOLE, l=0.3, k2=-20.0, num_steps=3),
        "kicker_thin": mk(E.KICKER, hkick=2e-4, vkick=-1e-4),
        "kicker_thick": mk(E.KICKER, l=0.2, hkick=2e-4, vkick=-1e-4, num_steps=1),
        "bend": mk(E.SBEND, l=2.0, g=0.0157),
        "bend_back": mk(E.SBEND, l=2.0, g=-0.0157),
        "bend_weak": mk(E.SBEND, l=0.5, g=0.002),
        "bend_k1": mk(E.SBEND, l=2.0, g=0.0157, k1=0.0135),
        "bend_k1_defocusing": mk(E.SBEND, l=2.0, g=0.0157, k1=-0.0135),
        "quad_offset": mk(E.QUADRUPOLE, l=0.3, k1=0.5, **off),
        "quad_corrector": mk(E.QUADRUPOLE, l=0.3, k1=0.5, hkick=1e-4, vkick=2e-4, num_steps=4, **off),
        "quad_corrector_straight": mk(E.QUADRUPOLE, l=0.3, k1=0.5, hkick=1e-4, num_steps=1),
        "sext_offset": mk(E.SEXTUPOLE, l=0.2, k2=20.0, num_steps=1, **off),
        "quad_pitch": mk(E.QUADRUPOLE, l=0.3, k1=0.5, x_pitch=1e-3, **off),
    }


def _beam(bmx, n, seed):
    """Angles of some 8 mrad, positions across the apertures, pz wide
    enough for both sides of the quadrupole series' limits, and a few particles at the zero orbit."""
    L = bmx.lattices
    sig = np.array([4e-3, 8e-3, 3e-3, 8e-3, 1e-3, 3e-2])
    b = L.gaussian_beam(n, seed=seed, sigma=sig)
    for i, s in enumerate((0.0, 1e-12, 5e-10)):
        if n > 100:
            for k in P.COORDS:
                b[k][7 + 64 * i] = s
    p0c, et = L.reference()
    b["beta"] = L.init_beta(b["pz"], p0c, et)
    return b


def _turn(bmx, ctx, arr, beam, how):
    """One pass through all elements: the generic or the cell kernel, the span kernel, the element
    kernel, or the recording one."""
    T = bmx.tracking
    lat = T.Lattice(ctx, arr)
    if how == "cell":
        assert lat.specialize()
    b = T.Beam.from_host(ctx, beam)
    n = len(arr)
    if how in ("turns", "cell"):
        T.track_beam(ctx, lat, b, 1, 0)
    elif how == "spans":  # cut inside blocks and round the end
        T.track_bunch(ctx, lat, b, 0, 5, 0)
        T.track_bunch(ctx, lat, b, 5, n - 3, 0)
        T.track_bunch(ctx, lat, b, n - 3, n, 0)
    elif how == "elements":
        for e in range(1, n + 1):
            T.track1_bunch(ctx, lat, b, e, 0)
    else:
        T.track_orbit(ctx, lat, b)
    ctx.synchronize()
    out = b.download()
    b.close()
    lat.close()
    return out


@pytest.mark.parametrize("ap", ["none", "ellipse", "rectangle", "off_axis"])
def test_single_elements(bmx, oracle, ctx, ap):
    """Each element, between two drifts: losses identical to the restatement, survivors within the
    per-element bar, 1e-12 for each of the three."""
    for name, e in _elements(bmx, **_apertures(bmx)[ap]).items():
        E = bmx.elements
        p0c, et = bmx.lattices.reference()
        d = E.make_element(E.DRIFT, p0c, et, l=0.5)
        arr = E.to_array([d, e, d])
        beam = _beam(bmx, 3001, 5)
        ref = P.copy_beam(beam)
        oracle.track_bunch(arr, ref, 1)
        print(f"operations {ap} {name}", flush=True)
        out = _turn(bmx, ctx, arr, beam, "turns")
        bad = P.loss_mismatch(out, ref)
        assert bad.size == 0, (name, bad[:5])
        err = P.rel_err(out, ref, ref["state"] == 1)
        assert err <= 3e-12, (name, err)


def _mixed_ring(bmx, cells=4):
    """A line of repeated cells of every kind of operation, each element of strengths of its own."""
    e = _elements(bmx, x_limit=0.02, y_limit=0.02, aperture_type=bmx.elements.APERTURE_ELLIPTICAL)
    cell = [e["drift"], e["quad_weak"], e["sext_1"], e["marker"], e["kicker_thick"], e["bend"], e["quad_mid"],
            e["quad_corrector"], e["sext_3"], e["bend_k1"], e["drift"], e["kicker_thin"], e["sext_offset"],
            e["bend_back"], e["quad_offset"], e["drift"]]
    arr = bmx.elements.to_array(cell * cells)
    # weak enough that a part of the beam gets through
    weak = arr["key"] != bmx.elements.SBEND
    arr["k1"][weak] *= 0.4
    arr["k2"] *= 0.3
    arr["hkick"] *= 0.1
    arr["vkick"] *= 0.1
    rng = np.random.default_rng(31)
    for f in ("k1", "k2", "g", "hkick", "vkick", "x_offset", "y_offset"):
        arr[f] *= 1 + 0.1 * rng.uniform(-1, 1, len(arr))
    return arr


@pytest.mark.parametrize("n", [1, 63, 65, 1000])
def test_kernels_give_the_same_bits(bmx, oracle, ctx, n):
    """The turn, span, element and recording kernels and the cell kernel agree: the same loss records,
    the restatement's, and the same bits for every survivor."""
    arr = _mixed_ring(bmx)
    beam = _beam(bmx, n, 9)
    for k, s in (("x", 0.2), ("y", 0.2), ("px", 0.02), ("py", 0.02), ("pz", 0.1)):
        beam[k] *= s
    ref = P.copy_beam(beam)
    oracle.track_bunch(arr, ref, 1)
    print(f"operations bits n={n}", flush=True)
    want = _turn(bmx, ctx, arr, beam, "turns")
    assert P.loss_mismatch(want, ref).size == 0
    if n == 1000:
        assert 20 < (ref["state"] != 1).sum() < 980
    alive = ref["state"] == 1
    for how in ("spans", "elements", "record", "cell"):
        out = _turn(bmx, ctx, arr, beam, how)
        assert P.loss_mismatch(out, want).size == 0, how
        for k in P.COORDS:
            assert np.array_equal(out[k][alive], want[k][alive]), (how, k)


def test_results_do_not_depend_on_the_wave(bmx, ctx):
    """Particles tracked alone and among others that fail the operations' tests or sit at the zero
    orbit: the same bits."""
    arr = _mixed_ring(bmx)
    beam = _beam(bmx, 256, 13)
    for k, s in (("x", 0.3), ("y", 0.3), ("px", 0.05), ("py", 0.05)):
        beam[k] *= s
    print("operations wave independence", flush=True)
    for how in ("turns", "cell"):
        mixed = _turn(bmx, ctx, arr, beam, how)
        for i in (0, 7, 71, 135, 200, 255):
            one = _turn(bmx, ctx, arr, {k: v[i:i + 1].copy() for k, v in beam.items()}, how)
            for k in P.KEYS:
                assert np.array_equal(one[k][0:1], mixed[k][i:i + 1]), (how, i, k)


@pytest.mark.parametrize("rows", ["none", "pz", "bend", "all", "coefficients", "cells"])
def test_radiation_maps_with_zero_parts(bmx, oracle, ctx, rows):
    """Radiation maps whose zero rows and columns the operation leaves out, the same in every cell (also
    with single coefficients that are zero in some cells) or not ("cells"): damping and fluctuations of
    a ring of plain and gradient bends and offset quadrupoles, one turn, losses identical and
    survivors within the whole-turn bar of the restatement."""
    T = bmx.tracking
    E = bmx.elements
    e = _elements(bmx, **_apertures(bmx)["ellipse"])
    arr = E.to_array([e["drift"], e["bend"], e["quad_offset"], e["drift"], e["bend_k1"], e["sext_1"]] * 4)
    maps = R.lattice_maps(arr, bmx, damp=1e2, stoc=1e2)
    keep = {"none": [], "pz": [5], "bend": [0, 1, 4, 5]}.get(rows, [0, 1, 2, 3, 4, 5])
    drop = [i for i in range(6) if i not in keep]
    for f in ("damp_dmat", "stoc_mat"):
        maps[f][:, :, drop, :] = 0
        maps[f][:, :, :, drop] = 0
    maps["xfer_damp_vec"][:, :, drop] = 0
    maps["ref_orb"][...] = 1e-4
    if rows == "coefficients":
        maps["damp_dmat"][:12, :, 5, 0] = maps["damp_dmat"][:, :, 1, :3] = maps["xfer_damp_vec"][6:, :, 1] = 0
        maps["stoc_mat"][6:, :, 4, 2] = maps["stoc_mat"][:, :, 3, 3] = 0
    if rows == "cells":
        maps["damp_dmat"][:6, :, 1, :] = maps["xfer_damp_vec"][:6, :, 1] = maps["stoc_mat"][:6, :, 2, :] = 0
    beam = _beam(bmx, 2000, 17)
    for k, s in (("x", 0.3), ("y", 0.3), ("px", 0.05), ("py", 0.05)):
        beam[k] *= s
    cfg = T.rad_config(damping=True, fluctuations=True, scale=1.25, seed=77)
    ocfg = oracle.RadConfig(1, 1, 0, 0, 1.25, 77)
    ref = P.copy_beam(beam)
    oracle.track_bunch(arr, ref, 1, rad_maps=maps, rad=ocfg)
    print(f"operations radiation rows={rows}", flush=True)
    lat = T.Lattice(ctx, arr, rad_maps=maps, rad=cfg)
    outs = []
    for special in (False, True):
        if special:
            assert lat.specialize()
        b = T.Beam.from_host(ctx, beam)
        T.track_beam(ctx, lat, b, 1, 0)
        ctx.synchronize()
        outs.append(b.download())
        b.close()
    lat.close()
    assert P.loss_mismatch(outs[0], ref).size == 0
    assert P.rel_err(outs[0], ref, ref["state"] == 1) <= 1e-11
    for k in P.KEYS:
        assert np.array_equal(outs[0][k], outs[1][k]), k


@pytest.mark.parametrize("sigma", [0.012, 0.025, 0.1])
def test_angles_about_the_operations_bound(bmx, oracle, ctx, sigma):
    """Drifts, sextupoles and bends at angles on both sides of the operations' bound (44 mrad) and far
    beyond it: losses identical to the restatement, survivors within the per-element bar, 1e-12 for
    each of the three elements, and the same bits from the element kernel for the particles on
    operations."""
    E = bmx.elements
    p0c, et = bmx.lattices.reference()
    d = E.make_element(E.DRIFT, p0c, et, l=0.5)
    e = _elements(bmx)
    beam = _beam(bmx, 3001, 23)
    rng = np.random.default_rng(29)
    for k in ("px", "py"):
        beam[k] = sigma * rng.standard_normal(3001)
    within = np.hypot(beam["px"], beam["py"]) < 0.04 * (1 + beam["pz"])
    for name in ("drift", "sext_1", "sext_3", "bend", "bend_back"):
        arr = E.to_array([d, e[name], d])
        ref = P.copy_beam(beam)
        oracle.track_bunch(arr, ref, 1)
        print(f"operations angles {name} {sigma}", flush=True)
        out = _turn(bmx, ctx, arr, beam, "turns")
        assert P.loss_mismatch(out, ref).size == 0, name
        assert P.rel_err(out, ref, ref["state"] == 1) <= 3e-12, name
        one = _turn(bmx, ctx, arr, beam, "elements")
        for k in P.COORDS:
            assert np.array_equal(out[k][within], one[k][within]), (name, k)
