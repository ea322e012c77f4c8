"""The axis-by-axis form of the phase contraction (k_axis_rot, k_axis_ab,
k_axis_pair, k_axis_pair_q) against the oracle where its tiles and rules can go
wrong: every kernel variant (bands, branches), meshes with three different
lengths, odd ones and ones beyond 31 points (two row tiles), cells beyond 7 along an
axis (four K steps), windows that leave lines short or empty, more than one round of
work items, polar terms, mesh_ref 2, states of a k split over calls.  Every case runs in the
form that the plan chose, which has to be this one (plan.form()), and as one product over all
cells.  Counts exact, exact zeros
equal, |g|^2 relative above 1e-6 * max within 1e-12 (FP64: sums of at most 1e3
terms of one sign pattern, a few hundred units of 1.1e-16 after the cancellation
the floor allows) and 1e-5 (mixed)."""
import types

import numpy as np
import pytest

from elphbolt_amd import interactions, synth
from elphbolt_amd._lib import ElphError
from elphbolt_amd.wannier import Wannier
from oracle import oracle as O

pytestmark = pytest.mark.gpu

FLOOR = 1e-6


def _rel(x, ref):
    x, ref = np.asarray(x).ravel(), np.asarray(ref).ravel()
    sel = np.abs(ref) > FLOOR * np.abs(ref).max()
    return float(np.max(np.abs(x[sel] - ref[sel]) / np.abs(ref[sel]))) if sel.any() else 0.0


def _material(nb, nat, ws, mesh, biw, polar=None, mesh_ref=1, seed=5):
    masses = [28.0855, 12.0107, 15.999, 24.305, 69.723, 74.92, 10.81, 30.97][:nat]
    mat = synth.make_material(f"axis_nb{nb}_na{nat}", 4.36, masses, nb, ws, mesh, seed, mesh_ref=mesh_ref,
                              bands_in_window=biw)
    return synth.with_polar(mat, polar, seed=3) if polar else mat


def _state(mat):
    o = O.Wannier(mat)
    eye = np.eye(3).ravel()  # one operation: meshes with different lengths keep no rotation
    el = O.Electrons(o, eye, 1, mat.wvmesh, mat.enref, mat.fsthick)
    ph = O.Phonons(o, eye, 1, mat.phmesh)
    return o, el, ph


# name, nb, nat, ws, mesh, bands in window, polar, precision
CASES = [
    ("nb8_na2", 8, 2, [5, 5, 5], [14, 16, 9], 3.0, None, "fp64"),
    ("nb8_na2_mixed", 8, 2, [5, 5, 5], [14, 16, 8], 3.0, None, "mixed"),
    ("nb8_na2_wide", 8, 2, [4, 4, 4], [24, 7, 8], 7.5, None, "fp64"),    # more than 64 items on a line
    ("nb7_na2_narrow", 7, 2, [6, 6, 6], [14, 16, 9], 0.4, None, "fp64"),  # short and missing lines
    ("nb3_na1", 3, 1, [4, 4, 4], [11, 13, 10], 1.5, None, "fp64"),
    ("nb8_na2_polar", 8, 2, [5, 5, 5], [13, 12, 9], 3.0, "sic", "fp64"),
    ("nb5_na3", 5, 3, [4, 4, 4], [12, 11, 9], 2.0, None, "fp64"),
    ("nb5_na3_polar_mixed", 5, 3, [7, 7, 7], [24, 20, 12], 2.0, "random", "mixed"),
    ("nb11_na3", 11, 3, [4, 4, 4], [12, 11, 9], 2.0, None, "fp64"),
    ("nb13_na4", 13, 4, [4, 4, 4], [12, 11, 9], 2.0, None, "fp64"),
    ("nb16_na5_polar", 16, 5, [4, 4, 4], [12, 11, 8], 2.0, "random", "fp64"),
    ("nb19_na2", 19, 2, [4, 4, 4], [12, 11, 8], 2.0, None, "fp64"),
    ("nb26_na8", 26, 8, [4, 4, 4], [24, 11, 8], 1.0, None, "fp64"),
    ("n0_34", 4, 2, [5, 5, 5], [34, 6, 6], 2.0, None, "fp64"),
    ("n1_33", 4, 2, [4, 4, 4], [12, 33, 4], 2.0, None, "fp64"),
    ("n0_62_n1_61", 2, 1, [5, 5, 5], [62, 61, 2], 1.0, None, "fp64"),
    ("r0_beyond_7", 4, 1, [24, 3, 3], [24, 10, 8], 2.0, None, "fp64"),
    ("r1_beyond_7", 4, 1, [3, 24, 3], [13, 24, 8], 2.0, None, "fp64"),
    ("n0_40_r0_beyond_7", 4, 1, [24, 3, 3], [40, 10, 8], 2.0, None, "fp64"),
    ("n1_40_r1_beyond_7", 4, 1, [3, 24, 3], [13, 40, 8], 2.0, None, "fp64"),
    ("r2_long", 4, 1, [3, 3, 15], [12, 13, 24], 2.0, None, "fp64"),
]


@pytest.mark.parametrize("name,nb,nat,ws,mesh,biw,polar,precision", CASES, ids=[c[0] for c in CASES])
def test_ibzk_axis(name, nb, nat, ws, mesh, biw, polar, precision):
    mat = _material(nb, nat, ws, mesh, biw, polar)
    _reaches(name, mat.rcells_q)
    o, el, ph = _state(mat)
    plan = interactions.IbzkPlan(Wannier(mat), el, ph, precision=precision)
    chosen = plan.form()
    assert chosen == (True, precision == "fp64" and mat.nwsk > 93)  # sums at the points of 93 cells: product
    # the in-window states of the first, a middle and the last k, over the first and last rows
    act = np.abs(el.ens_irred - el.enref) <= el.fsthick
    ks = np.nonzero(act.any(1))[0]
    nwin = (np.abs(el.ens - el.enref) <= el.fsthick).sum(1)
    offs = np.concatenate([[0], np.cumsum(nwin)]) * mat.nbr
    span = min(el.nwv, 48 if nb <= 8 else 20)
    err = {}
    for ik in sorted({int(ks[0]), int(ks[len(ks) // 2]), int(ks[-1])}):
        first, last = ik * nb + 1, (ik + 1) * nb
        refs = [(r0, O.ibzk_g2_window(o, el, ph, first, last, r0 + 1, span)) for r0 in (0, el.nwv - span)]
        for form in ((False, False), chosen):
            print(f"axis ibzk {name} {precision}: k {ik + 1}, {el.nwv} rows, form {form}", flush=True)
            assert plan.form(*form) == form
            c_g, g_g = plan.run(first, last)
            for r0, (c_o, g_o, _) in refs:
                got = g_g[:, offs[r0]:offs[r0 + span]]
                sel = c_o >= 0
                assert np.array_equal(sel, c_g >= 0) and sel.any()
                assert np.all(c_g[sel] == plan.nprocs)
                ref = g_o[sel][:, :got.shape[1]]
                assert np.array_equal(ref == 0.0, got[sel] == 0.0)
                err[form] = max(err.get(form, 0.0), _rel(got[sel], ref))
    print(f"  max rel {err}", flush=True)
    assert max(err.values()) < (1e-12 if precision == "fp64" else 1e-5)
    # the same bits whatever states share a call
    one = plan.run(int(ks[0]) * nb + 1, int(ks[-1]) * nb + nb) if len(ks) < 40 else None
    if one is not None:
        assert np.array_equal(one[1][-nb:], g_g)


def test_ibzk_axis_mesh_ref2():
    """The oracle takes, as the phonons of the electron mesh, the given ones on
    the phonon mesh and the library's own ph_wann off it (the phonons the plan
    interpolates), so both sides rotate with the same eigenvectors."""
    mat = _material(4, 2, [5, 5, 5], [14, 12, 10], 2.0, mesh_ref=2)
    o, el, ph = _state(mat)
    w = Wannier(mat)
    mesh = np.asarray(mat.wvmesh)
    i = np.arange(int(np.prod(mesh)))
    pts = np.stack([i % mesh[0], (i // mesh[0]) % mesh[1], i // (mesh[0] * mesh[1])], 1)
    ens, evecs, _ = w.ph_wann(pts / mesh)
    on = np.all(pts % 2 == 0, axis=1)
    half, cm = pts[on] // 2, mesh // 2
    coarse = (half[:, 2] * cm[1] + half[:, 1]) * cm[0] + half[:, 0]
    ens[on], evecs[on] = ph.ens[coarse], ph.evecs[coarse]
    fine = types.SimpleNamespace(wvmesh=mesh, nwv=len(pts), ens=ens, evecs=evecs, nwv_irred=len(pts),
                                 indexlist_irred=np.arange(1, len(pts) + 1))
    last = 8
    c_o, g_o = O.ibzk_g2(o, el, fine, 1, 1, last)
    plan = interactions.IbzkPlan(w, el, ph, mesh_ref=2, precision="fp64")
    assert plan.form() == (True, True)
    act = c_o >= 0
    for form in ((True, True), (False, False)):
        assert plan.form(*form) == form
        c_g, g_g = plan.run(1, last)
        assert np.array_equal(c_o, c_g) and act.any()
        assert np.array_equal(g_o[act] == 0.0, g_g[act] == 0.0)
        assert _rel(g_g[act], g_o[act]) < 1e-12


# name, nb, nat, ws, mesh, bands in window, polar
CASES_Q = [
    ("nb6_na2", 6, 2, [4, 4, 4], [12, 11, 9], 2.5, None),
    ("nb8_na1_narrow", 8, 1, [5, 5, 5], [14, 13, 9], 0.6, None),
    ("nb8_na1_wide", 8, 1, [4, 4, 4], [24, 7, 8], 7.5, None),
    ("nb11_na2_polar", 11, 2, [4, 4, 4], [12, 11, 9], 2.0, "sic"),
    ("nb14_na1", 14, 1, [4, 4, 4], [12, 11, 9], 2.0, None),
    ("nb19_na1", 19, 1, [4, 4, 4], [24, 11, 8], 2.0, None),
    ("n0_35_n1_33", 4, 1, [5, 5, 5], [35, 33, 2], 1.5, None),
    ("r0_beyond_7", 4, 1, [24, 3, 3], [24, 10, 8], 2.0, None),
]


def _reaches(name, cells):
    """Cases named for cells beyond 7 along an axis have them (four K steps; k_axis_pts beyond 7 along R0)."""
    for axis in (0, 1):
        if f"r{axis}_beyond_7" in name:
            assert np.abs(np.asarray(cells)[:, axis]).max() > 7


@pytest.mark.parametrize("name,nb,nat,ws,mesh,biw,polar", CASES_Q, ids=[c[0] for c in CASES_Q])
def test_ibzq_axis(name, nb, nat, ws, mesh, biw, polar):
    mat = _material(nb, nat, ws, mesh, biw, polar, seed=6)
    _reaches(name, mat.rcells_k)
    o, el, ph = _state(mat)
    first = 3 * mat.nbr + 1  # past q = 0
    last = first + (mat.nbr if nb > 8 else 2 * mat.nbr) - 1
    print(f"axis ibzq {name}: states {first}..{last}, {el.nwv} rows", flush=True)
    c_o, g_o = O.ibzq_g2(o, el, ph, first, last)
    plan = interactions.IbzqPlan(Wannier(mat), el, ph)
    chosen = plan.form()
    assert chosen == (True, mat.nwsk > 93)
    for form in (chosen, (False, False)):
        assert plan.form(*form) == form
        c_g, g_g = plan.run(first, last)
        assert np.array_equal(c_o, c_g) and c_o.max() > 0
        err = 0.0
        for t, n in enumerate(c_o):
            assert np.array_equal(g_o[t, :n] == 0.0, g_g[t, :n] == 0.0)
            err = max(err, _rel(g_g[t, :n], g_o[t, :n]))
        print(f"  form {form}: max rel {err:.2e}", flush=True)
        assert err < 1e-12


@pytest.mark.parametrize("kind", ["ibzk", "ibzq"])
def test_many_points_per_pass(kind):
    """More IBZ points than one pass of the mesh-point sum takes (1024), more than its
    8 planes and 64 lines at a time: a run into device rows, which takes the large
    groups, gives the bits of runs into host rows, which take groups of 64."""
    mat = _material(3, 1, [5, 5, 5], [14, 16, 9], 1.5)
    _, el, ph = _state(mat)
    w = Wannier(mat)
    plan = (interactions.IbzkPlan if kind == "ibzk" else interactions.IbzqPlan)(w, el, ph)
    assert plan.form() == (True, True)
    assert (el.nwv_irred if kind == "ibzk" else ph.nwv_irred) > 1024
    nst = (el if kind == "ibzk" else ph).nwv_irred * 3
    width = plan.nprocs if kind == "ibzk" else plan.stride
    print(f"axis {kind}: {nst} states in one call", flush=True)
    dev = w.device_buffer((nst, width))
    counts, _ = plan.run(1, nst, out=dev)
    rows = dev.numpy()
    for first, last in [(1, 60), (3 * 1000 + 2, 3 * 1060), (nst - 40, nst)]:
        c, g = plan.run(first, last)
        assert np.array_equal(c, counts[first - 1:last]) and c.max() > 0
        got = rows[first - 1:last]
        if kind == "ibzk":
            assert np.array_equal(got[c >= 0], g[c >= 0])
        else:
            for t, n in enumerate(c):
                assert np.array_equal(got[t, :n], g[t, :n])
    # the form that a run takes when the device has no room for the large groups
    assert plan.small(True) and plan.form() == (True, True)
    few = w.device_buffer((nst, width))
    c, _ = plan.run(1, nst, out=few)
    assert np.array_equal(c, counts)
    part = few.numpy()
    for t in np.flatnonzero(c > 0):
        assert np.array_equal(part[t, :c[t]], rows[t, :c[t]])
    assert not plan.small(False)


def test_batch_of_both_forms():
    """Two plans of one size class, the first in this form: the other still has its tile shape timed, a
    change of the point sum after a plan was added takes effect, and the replayed rows are the plans' own."""
    mat = _material(4, 2, [5, 5, 5], [14, 12, 10], 2.0)
    _, el, ph = _state(mat)
    w = Wannier(mat)
    plans = [interactions.IbzkPlan(w, el, ph) for _ in range(2)]
    assert plans[0].form() == (True, True) and plans[1].form(pair=False) == (False, True)
    b = interactions.Batch(nstreams=2)
    last = 40 * mat.nb
    outs = [b.add(p, 1, last) for p in plans]
    plans[0].form(points=False)
    b.prepare(autotune=True)
    cls = {c["path"]: c for c in b.classes()}
    print("batch of both forms", cls, flush=True)
    assert len(cls) == 2 and cls[2]["members"] == 1 and cls[2]["candidates"] == 1
    tiles = cls[0] if 0 in cls else cls[1]
    assert tiles["members"] == 1 and tiles["candidates"] > 1
    eager = []
    for p, form in zip(plans, ((True, False), (False, True))):
        assert p.form() == form
        c, g = p.run(1, last)
        eager.append(g[c >= 0])
    for _ in range(2):
        assert b.run() > 0
        for (c, out), g in zip(outs, eager):
            assert np.array_equal(out.numpy(), g)
        w.synchronize()
    b.close()


# kind, nb, nat, ws, mesh, bands in window, precision: the axis sums have 1/10, 1/2.2, 1/2.8 of the
# product's multiply-adds, and took longer on plans of these shapes (second tile of q; branches; short lines)
SLOWER = [
    ("ibzk", 15, 1, [4, 4, 4], [60, 8, 8], 4.0, "mixed"),
    ("ibzk", 17, 5, [4, 4, 4], [6, 21, 15], 2.2, "fp64"),
    ("ibzk", 8, 1, [5, 5, 5], [35, 12, 10], 0.3, "fp64"),
    ("ibzq", 20, 2, [4, 4, 4], [7, 18, 8], 3.3, "fp64"),
]


@pytest.mark.parametrize("kind,nb,nat,ws,mesh,biw,precision", SLOWER, ids=[f"{c[0]}_nb{c[1]}_n0_{c[4][0]}" for c in SLOWER])
def test_product_kept_where_it_is_faster(kind, nb, nat, ws, mesh, biw, precision):
    mat = _material(nb, nat, ws, mesh, biw)
    _, el, ph = _state(mat)
    plan = (interactions.IbzkPlan if kind == "ibzk" else interactions.IbzqPlan)(Wannier(mat), el, ph, precision=precision)
    assert not plan.form()[0]


def test_form_of_a_plan():
    """A plan that does not have a form refuses it and keeps the one it has."""
    mat = synth.tiny(nb=4, natoms=2, ws=3, wv=4, seed=12)  # the sums cost as much as the product
    _, el, ph = _state(mat)
    w = Wannier(mat)
    plan = interactions.IbzkPlan(w, el, ph, precision="mixed")
    assert plan.form() == (False, False)
    for kw in (dict(pair=True), dict(points=True)):
        with pytest.raises(ElphError):
            plan.form(**kw)
    assert plan.form(pair=False) == (False, False)
