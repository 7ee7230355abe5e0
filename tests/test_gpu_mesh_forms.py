"""Meshes that the entry points accept besides those that the generator makes: an edge's
triangles on either side (a coastal edge whose only triangle is its second one), two edges
between the same nodes (a crack), a node with a second fan of triangles beside a closed one.
compute_w, the upwind step and the FCT step against the oracle, bit for bit (every per-node
sum runs in the oracle's (edge, side) order), and the backward to 1e-11 of its cotangents."""

import numpy as np
import pytest

from oracle import fct_numpy as O
from oracle import fct_vjp as V

pytestmark = pytest.mark.gpu


def _rebuilt(m, **changed):
    """The mesh with the given arrays in place of its own."""
    from fesom_jax_amd.mesh import MESH_ARRAY_FIELDS, MESH_META_FIELDS, mesh_from_arrays
    arrays = {k: np.array(changed.get(k, getattr(m, k))) for k in MESH_ARRAY_FIELDS}
    meta = {k: getattr(m, k) for k in MESH_META_FIELDS}
    meta["edge2D"] = len(arrays["edges"])
    return mesh_from_arrays(arrays, meta, check_orientation=False)


def _sides_swapped(m, which):
    """The edges ``which`` with their two triangles exchanged. An edge's flux is the first
    triangle's term minus the second one's, so the vectors change places and sign."""
    et, cr = m.edge_tri.copy(), m.edge_cross_dxdy.copy()
    et[which] = et[which][:, ::-1]
    cr[which] = -cr[which][:, [2, 3, 0, 1]]
    return _rebuilt(m, edge_tri=et, edge_cross_dxdy=cr)


def _coastal(m):
    c = np.zeros(m.nod2D, bool)
    c[m.edges[(m.edge_tri < 0).any(axis=1)].reshape(-1)] = True
    return c


def _cracked(m, count, seed):
    """``count`` interior edges between coastal nodes (whose fans are open), no two at one
    node, as two edges between the same nodes: the first keeps the first triangle, a new one
    at the end of the list has the second."""
    rng = np.random.default_rng(seed)
    deg = np.bincount(m.edges.reshape(-1), minlength=m.nod2D)
    coast = _coastal(m)
    seen, pick = set(), []
    for e in rng.permutation(np.nonzero((m.edge_tri >= 0).all(axis=1) & coast[m.edges].all(axis=1))[0]):
        a, b = m.edges[e]
        if len(pick) < count and a not in seen and b not in seen and max(deg[a], deg[b]) < 8:
            pick.append(e)
            seen.update((a, b))
    assert pick
    pick = np.array(pick)
    et, cr, ud = m.edge_tri.copy(), m.edge_cross_dxdy.copy(), m.edge_up_dn_tri.copy()
    more_et, more_cr = et[pick].copy(), cr[pick].copy()
    more_et[:, 0], more_cr[:, :2] = -1, 0.0
    et[pick, 1], cr[pick, 2:], ud[pick] = -1, 0.0, -1
    return _rebuilt(m, edges=np.r_[m.edges, m.edges[pick]], edge_tri=np.r_[et, more_et],
                    edge_cross_dxdy=np.r_[cr, more_cr], edge_up_dn_tri=np.r_[ud, ud[pick]],
                    edge_dxdy=np.r_[m.edge_dxdy, m.edge_dxdy[pick]])


def _pinched(m):
    """A coastal node joined to a node of five neighbours, which then has that open fan
    beside its closed one (such a node has no ring)."""
    deg = np.bincount(m.edges.reshape(-1), minlength=m.nod2D)
    coast = _coastal(m)
    near = lambda n: set(m.edges[(m.edges == n).any(axis=1)].reshape(-1)) - {n}
    for a in np.nonzero(~coast & (deg == 5))[0]:
        for b in np.nonzero(coast & (deg <= 3))[0]:
            if not near(a) & (near(b) | {b}):
                break
        else:
            continue
        break
    en, ed = m.elem_nodes.copy(), m.edges.copy()
    en[en == b], ed[ed == b] = a, a
    lev = {k: getattr(m, k).copy() for k in ("nlevels_nod2D", "nlevels_nod2D_min", "ulevels_nod2D",
                                             "ulevels_nod2D_max", "area", "areasvol")}
    for k, pick in (("nlevels_nod2D", max), ("nlevels_nod2D_min", min), ("ulevels_nod2D", min),
                    ("ulevels_nod2D_max", max)):
        lev[k][a] = pick(lev[k][a], lev[k][b])
        lev[k][b] = 1                             # (the number left over: no layer)
    for k in ("area", "areasvol"):
        lev[k][a] = np.maximum(lev[k][a], lev[k][b])
    order = np.argsort(en.reshape(-1), kind="stable")
    off = np.r_[0, np.cumsum(np.bincount(en.reshape(-1), minlength=m.nod2D))]
    return _rebuilt(m, elem_nodes=en, edges=ed, nod_in_elem2D=order // 3, nod_in_elem2D_offsets=off,
                    **lev)


def _mesh(form, nl, degree8):
    from fesom_jax_amd.meshgen import icosahedral_mesh
    m = icosahedral_mesh(3, nl, seed=51, degree8=degree8, min_levels=3, polar_cap_deg=60.0)
    coast = np.nonzero((m.edge_tri < 0).any(axis=1))[0]
    if form == "coast_second":
        return _sides_swapped(m, coast)
    if form == "sides_mixed":
        return _sides_swapped(m, np.nonzero(np.random.default_rng(52).random(m.edge2D) < 0.5)[0])
    if form == "cracked":
        return _cracked(m, 40, 53)
    return _pinched(m)


FORMS = [("coast_second", 48, 0), ("coast_second", 70, 10), ("sides_mixed", 48, 0),
         ("sides_mixed", 70, 10), ("cracked", 48, 0), ("cracked", 70, 10),
         ("pinched", 48, 0), ("pinched", 70, 10)]


@pytest.mark.parametrize("form,nl,degree8", FORMS)
def test_compute_w_and_upwind(form, nl, degree8, torch_dev):
    import torch
    from fesom_jax_amd.ale import compute_w
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.tracer_adv import advect_one, get_plan
    m = _mesh(form, nl, degree8)
    c = make_case(m, seed=54, dt=2700.0)
    assert get_plan(m, torch_dev).fused_available
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev)
    print(f"[forms] {form} N={m.nod2D} D={m.edge2D} nl={nl}", flush=True)
    w = compute_w(m, t(c["uv"]), t(c["helem"])).cpu().numpy()
    assert np.array_equal(w, O.compute_w(m, c["uv"], c["helem"]))
    T = np.nan_to_num(c["T"][0])       # (a node without triangles has no smoothed field)
    To = 0.98 * T + 0.3
    flow = [c[k] for k in ("uv", "w_e", "helem", "hnode", "hnode_new")]
    got, _ = advect_one(m, *map(t, flow), t(T), t(To), dt=c["dt"])
    want, _ = O.advect_one(m, *flow, T, To, dt=c["dt"])
    assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("form", [0, 1])
def test_compute_w_without_rings(form, torch_dev):
    """Both forms of the divergence on a mesh that has node tables and no rings."""
    import torch
    from fesom_jax_amd import _lib
    from fesom_jax_amd.ale import compute_w
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.tracer_adv import get_plan
    for nl in (48, 70):
        m = _mesh("pinched", nl, 0)
        c = make_case(m, seed=55, dt=2700.0)
        plan = get_plan(m, torch_dev)
        _lib.check(plan.lib.fct_plan_set_tuning(plan.ptr, _lib.FCT_TUNE_W_EDGE_FLUX, form), "tuning")
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev)
        w = compute_w(m, t(c["uv"]), t(c["helem"])).cpu().numpy()
        assert np.array_equal(w, O.compute_w(m, c["uv"], c["helem"])), nl


@pytest.mark.parametrize("form,nl,degree8", FORMS)
def test_step_and_backward(form, nl, degree8, torch_dev):
    """(On a pinched mesh the backward takes the flat kernels.)"""
    import torch
    from fesom_jax_amd.adjoint import advect_fct_vjp
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.tracer_adv import advect_one_fct
    m = _mesh(form, nl, degree8)
    c = make_case(m, seed=56, dt=2700.0)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev)
    T = np.nan_to_num(c["T"][0])
    To = 0.98 * T + 0.3
    flow = [c[k] for k in ("uv", "w_e", "helem", "hnode", "hnode_new")]
    got, _ = advect_one_fct(m, *map(t, flow), t(T), t(To), dt=c["dt"])
    want = O.advect_one_fct(m, *flow, T, To, dt=c["dt"])[0]
    assert np.array_equal(got.cpu().numpy(), want)
    g = np.random.default_rng(57).standard_normal(T.shape)
    gT, gTo, guv, gw = advect_fct_vjp(m, *map(t, flow), [t(T)], [t(To)], [t(g)], dt=c["dt"])
    want = V.advect_one_fct_vjp(m, *flow, T, To, g, dt=c["dt"])
    for name, a, b in zip(("g_T", "g_T_old", "g_uv", "g_w"), (gT[0], gTo[0], guv, gw), want):
        a = a.cpu().numpy()
        assert np.abs(a - b).max() <= 1e-11 * max(np.abs(b).max(), 1e-300), name
