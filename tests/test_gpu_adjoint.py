"""GPU adjoint (fct_backward) against the CPU reverse-mode oracle (oracle/fct_vjp.py),
which is itself pinned by finite differences (tests/test_oracle_vjp.py). Tolerance:
normwise relative difference <= 1e-11 per cotangent (accumulation orders differ from
the oracle's, so the results agree to rounding, not bit for bit)."""

import numpy as np
import pytest

from conftest import sharp_case
from oracle import fct_numpy as O
from oracle import fct_vjp as V

pytestmark = pytest.mark.gpu

TOL = 1e-11


def _rel(a, b):
    den = max(float(np.abs(b).max()), 1e-300)
    return float(np.abs(a - b).max()) / den


def _oracle(mesh, c, Ts, Tos, gs, **opts):
    out = [V.advect_one_fct_vjp(mesh, c["uv"], c["w_e"], c["helem"], c["hnode"],
                                c["hnode_new"], T, To, g, dt=c["dt"], **opts)
           for T, To, g in zip(Ts, Tos, gs)]
    res = ([o[0] for o in out], [o[1] for o in out], sum(o[2] for o in out),
           sum(o[3] for o in out))
    return res + ((sum(o[4] for o in out),) if opts.get("w_i") is not None else ())


def _gpu(mesh, c, Ts, Tos, gs, dev, **opts):
    import torch
    from fesom_jax_amd.adjoint import advect_fct_vjp
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    opts = {k: (None if v is None else t(v)) for k, v in opts.items()}
    out = advect_fct_vjp(mesh, t(c["uv"]), t(c["w_e"]), t(c["helem"]), t(c["hnode"]),
                         t(c["hnode_new"]), [t(x) for x in Ts], [t(x) for x in Tos],
                         [t(x) for x in gs], dt=c["dt"], **opts)
    torch.cuda.synchronize()
    gT, gTo = out[0], out[1]
    return ([x.cpu().numpy() for x in gT], [x.cpu().numpy() for x in gTo]) + \
        tuple(x.cpu().numpy() for x in out[2:])


def _compare(name, got, want):
    gT, gTo, guv, gw = got[:4]
    wT, wTo, wuv, ww = want[:4]
    assert len(got) == len(want)
    for j in range(len(gT)):
        assert _rel(gT[j], wT[j]) <= TOL, (name, "g_T", j, _rel(gT[j], wT[j]))
        assert _rel(gTo[j], wTo[j]) <= TOL, (name, "g_T_old", j, _rel(gTo[j], wTo[j]))
    assert _rel(guv, wuv) <= TOL, (name, "g_uv", _rel(guv, wuv))
    assert _rel(gw, ww) <= TOL, (name, "g_w", _rel(gw, ww))
    if len(got) > 4:
        assert _rel(got[4], want[4]) <= TOL, (name, "g_w_i", _rel(got[4], want[4]))


def _split(mesh, c, seed):
    """An implicit split w_i of both signs and a moving-level stencil (Z3d, zbar3)."""
    rng = np.random.default_rng(seed)
    wm = mesh.node_iface_mask
    w_i = np.where(wm, 0.3 * np.abs(c["w_e"]).max() * rng.standard_normal(wm.shape), 0.0)
    zb3 = mesh.zbar_3d_n * (1.0 + 0.01 * rng.random(mesh.zbar_3d_n.shape))
    Z3d = np.concatenate([0.5 * (zb3[:, :-1] + zb3[:, 1:]), zb3[:, -1:]], axis=1)
    return w_i, Z3d, zb3


def _cot(mesh, K, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((mesh.nod2D, mesh.nl)) for _ in range(K)]


def test_adjoint_pi_two_tracers(pi_mesh, pi_case, torch_dev):
    c = pi_case
    Ts = c["T"]
    Tos = [0.995 * T for T in Ts]
    gs = _cot(pi_mesh, 2, 1)
    _compare("pi", _gpu(pi_mesh, c, Ts, Tos, gs, torch_dev), _oracle(pi_mesh, c, Ts, Tos, gs))


def test_adjoint_pi_limiter_active(pi_mesh, pi_case, torch_dev):
    c = sharp_case(pi_mesh, pi_case, 2.0)
    gs = _cot(pi_mesh, 1, 2)
    Ts, Tos = c["T"][:1], c["T_old"][:1]
    _, _, p = O.advect_one_fct(pi_mesh, c["uv"], c["w_e"], c["helem"], c["hnode"],
                               c["hnode_new"], Ts[0], Tos[0], dt=c["dt"], return_parts=True)
    assert (p["plus_fac"][pi_mesh.node_layer_mask] < 1).mean() > 0.02
    _compare("pi sharp", _gpu(pi_mesh, c, Ts, Tos, gs, torch_dev),
             _oracle(pi_mesh, c, Ts, Tos, gs))


def test_adjoint_icosa_nl70(torch_dev):
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh
    m = icosahedral_mesh(3, 70, seed=51)
    c = make_case(m, seed=52, dt=2700.0)
    Ts = c["T"]
    Tos = [0.99 * T + 0.01 * T[::-1] for T in Ts]
    gs = _cot(m, 2, 3)
    _compare("icosa3 nl70", _gpu(m, c, Ts, Tos, gs, torch_dev), _oracle(m, c, Ts, Tos, gs))


def test_adjoint_is_deterministic(pi_mesh, pi_case, torch_dev):
    c = pi_case
    gs = _cot(pi_mesh, 2, 4)
    a = _gpu(pi_mesh, c, c["T"], c["T_old"], gs, torch_dev)
    b = _gpu(pi_mesh, c, c["T"], c["T_old"], gs, torch_dev)
    for x, y in zip(a[0] + a[1] + [a[2], a[3]], b[0] + b[1] + [b[2], b[3]]):
        assert np.array_equal(x, y)


def test_autograd_function_matches_vjp(pi_mesh, pi_case, torch_dev):
    import torch
    from fesom_jax_amd.adjoint import fct_step
    c = pi_case
    t = lambda a, rg=False: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev).requires_grad_(rg)
    uv, w = t(c["uv"], True), t(c["w_e"], True)
    T = [t(x, True) for x in c["T"]]
    To = [t(0.99 * x, True) for x in c["T"]]
    out = fct_step(pi_mesh, uv, w, t(c["helem"]), t(c["hnode"]), t(c["hnode_new"]), T, To,
                   dt=c["dt"])
    gs = _cot(pi_mesh, 2, 5)
    loss = sum((o * t(g)).sum() for o, g in zip(out, gs))
    grads = torch.autograd.grad(loss, [*T, *To, uv, w])
    want = _oracle(pi_mesh, c, c["T"], [0.99 * x for x in c["T"]], gs)
    for j in range(2):
        assert _rel(grads[j].cpu().numpy(), want[0][j]) <= TOL
        assert _rel(grads[2 + j].cpu().numpy(), want[1][j]) <= TOL
    assert _rel(grads[4].cpu().numpy(), want[2]) <= TOL
    assert _rel(grads[5].cpu().numpy(), want[3]) <= TOL


def test_rollout_gradient_matches_oracle_chain(torch_dev):
    """Four chained steps: torch autograd through FctStep against the oracle's
    reverse chain (T_old <- T, T <- T_new), loss on the surface level."""
    import torch
    from fesom_jax_amd.adjoint import rollout
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh
    m = icosahedral_mesh(3, 48, seed=61)
    c = make_case(m, seed=62, dt=2700.0)
    nsteps = 4
    rng = np.random.default_rng(7)
    target = [T + 0.2 * rng.standard_normal(T.shape) * m.node_layer_mask for T in c["T"]]
    surf = m.node_layer_mask[:, 0]
    # oracle: forward trajectory, then the reverse chain
    traj = [(list(c["T"]), list(c["T_old"]))]
    for _ in range(nsteps):
        T, To = traj[-1]
        Tn = [O.advect_one_fct(m, c["uv"], c["w_e"], c["helem"], c["hnode"], c["hnode_new"],
                               T[j], To[j], dt=c["dt"])[0] for j in range(2)]
        traj.append((Tn, T))
    gT = [np.zeros_like(x) for x in c["T"]]
    for j in range(2):
        gT[j][:, 0] = np.where(surf, 2.0 * (traj[-1][0][j][:, 0] - target[j][:, 0]), 0.0)
    gTo = [np.zeros_like(x) for x in c["T"]]
    guv = np.zeros_like(c["uv"])
    for s in range(nsteps - 1, -1, -1):
        T, To = traj[s]
        res = [V.advect_one_fct_vjp(m, c["uv"], c["w_e"], c["helem"], c["hnode"],
                                    c["hnode_new"], T[j], To[j], gT[j], dt=c["dt"])
               for j in range(2)]
        guv = guv + sum(r[2] for r in res)
        # T_s feeds step s (as T) and step s+1 (as T_old)
        gT, gTo = [r[0] + gTo[j] for j, r in enumerate(res)], [r[1] for r in res]
    want_T0 = [gT[j] for j in range(2)]
    want_To0 = gTo
    # GPU: autograd through the rollout
    t = lambda a, rg=False: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev).requires_grad_(rg)
    uv = t(c["uv"], True)
    T0 = [t(x, True) for x in c["T"]]
    To0 = [t(x, True) for x in c["T_old"]]
    fin = rollout(m, uv, t(c["w_e"]), t(c["helem"]), t(c["hnode"]), t(c["hnode_new"]), T0,
                  To0, nsteps, dt=c["dt"])
    sm = t(surf.astype(np.float64))
    loss = sum((((f[:, 0] - t(tg[:, 0])) ** 2) * sm).sum() for f, tg in zip(fin, target))
    grads = torch.autograd.grad(loss, [*T0, *To0, uv])
    for j in range(2):
        assert _rel(grads[j].cpu().numpy(), want_T0[j]) <= 1e-10
        assert _rel(grads[2 + j].cpu().numpy(), want_To0[j]) <= 1e-10
    assert _rel(grads[4].cpu().numpy(), guv) <= 1e-10


def test_backward_rejects_unsupported(pi_mesh, pi_case, torch_dev):
    import torch
    from fesom_jax_amd.adjoint import advect_fct_vjp
    c = pi_case
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev)
    with pytest.raises(ValueError):
        advect_fct_vjp(pi_mesh, t(c["uv"]), t(c["w_e"]), t(c["helem"]), t(c["hnode"]),
                       t(c["hnode_new"]), [t(c["T"][0])], [t(c["T_old"][0])], [], dt=c["dt"])


@pytest.mark.parametrize("kind", ["w_i", "Z3d", "both"])
def test_adjoint_split_and_zstar(kind, torch_dev):
    """The implicit split (the Thomas solve reversed, w_e + w_i in adf_v, g_w_i) and the
    moving-level QR4C stencil, smooth and limiter-active."""
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh
    m = icosahedral_mesh(3, 48, seed=41)
    c0 = make_case(m, seed=42, dt=2700.0)
    for sharp in (False, True):
        c = sharp_case(m, c0, 2.0) if sharp else c0
        w_i, Z3d, zb3 = _split(m, c, 7)
        opts = {"w_i": dict(w_i=w_i), "Z3d": dict(Z3d=Z3d, zbar3=zb3),
                "both": dict(w_i=w_i, Z3d=Z3d, zbar3=zb3)}[kind]
        Ts, Tos = c["T"][:2], [0.99 * T + 0.01 * T[::-1] for T in c["T"][:2]]
        if sharp:
            Tos = c["T_old"][:2]
        gs = _cot(m, len(Ts), 3)
        print(f"[adjoint] {kind} sharp={sharp}", flush=True)
        _compare(f"{kind} sharp={sharp}", _gpu(m, c, Ts, Tos, gs, torch_dev, **opts),
                 _oracle(m, c, Ts, Tos, gs, **opts))


def test_adjoint_split_pi(pi_mesh, pi_case, torch_dev):
    c = pi_case
    w_i, Z3d, zb3 = _split(pi_mesh, c, 17)
    Ts, Tos, gs = c["T"][:1], [0.995 * c["T"][0]], _cot(pi_mesh, 1, 18)
    opts = dict(w_i=w_i, Z3d=Z3d, zbar3=zb3)
    _compare("pi split", _gpu(pi_mesh, c, Ts, Tos, gs, torch_dev, **opts),
             _oracle(pi_mesh, c, Ts, Tos, gs, **opts))


@pytest.mark.parametrize("level,nl,degree8,scattered,K,split", [
    (2, 12, 0, False, 1, False), (3, 64, 0, True, 2, False), (3, 65, 0, False, 2, True),
    (4, 70, 20, False, 1, True), (4, 48, 20, True, 3, False), (3, 128, 0, False, 1, True),
    (3, 23, 0, False, 5, True)])
def test_column_adjoint_forms(level, nl, degree8, scattered, K, split, torch_dev):
    """The wavefront-per-column backward over the meshes it takes: nl at and either side
    of the 64-lane slot and at its largest, 6- and 8-slot tables, scattered numbering,
    more tracers than the plan has slots (5 of 4), with the limiter active; the oracle's
    cotangents to the module's tolerance."""
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh, shuffled
    m = icosahedral_mesh(level, nl, seed=101, degree8=degree8)
    if scattered:
        m = shuffled(m, 102)
    c = sharp_case(m, make_case(m, seed=103, dt=2700.0), 1.5)
    Ts = [c["T"][0] * (1.0 + 0.1 * j) for j in range(K)]
    Tos = [c["T_old"][0] + 0.2 * j for j in range(K)]
    opts = {}
    if split:
        w_i, Z3d, zb3 = _split(m, c, 104)
        opts = dict(w_i=w_i, Z3d=Z3d, zbar3=zb3)
    gs = _cot(m, K, 105)
    _compare(f"icosa{level} nl{nl}", _gpu(m, c, Ts, Tos, gs, torch_dev, **opts),
             _oracle(m, c, Ts, Tos, gs, **opts))


def test_flat_adjoint_of_long_columns(torch_dev):
    """Meshes that the column kernels do not take (nl > 128) keep the flat backward."""
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh
    m = icosahedral_mesh(2, 130, seed=106)
    c = sharp_case(m, make_case(m, seed=107, dt=2700.0), 1.5)
    w_i, Z3d, zb3 = _split(m, c, 108)
    gs = _cot(m, 2, 109)
    Ts, Tos = [c["T"][0], 1.1 * c["T"][0]], [c["T_old"][0]] * 2
    for opts in ({}, dict(w_i=w_i, Z3d=Z3d, zbar3=zb3)):
        _compare("icosa2 nl130", _gpu(m, c, Ts, Tos, gs, torch_dev, **opts),
                 _oracle(m, c, Ts, Tos, gs, **opts))


@pytest.mark.parametrize("level,nl,degree8,K,split", [
    (2, 13, 0, 2, True), (3, 65, 10, 3, True), (3, 47, 0, 4, False), (3, 31, 0, 5, False),
    (6, 31, 0, 2, False), (6, 34, 20, 3, True), (6, 66, 0, 2, False)])
def test_adjoint_two_tracers_per_launch(level, nl, degree8, K, split, torch_dev):
    """Small meshes reverse two tracers per launch: against a plan with one tracer slot,
    which reverses them one after the other, bit for bit. Odd N * L (workspace alignment),
    a last tracer alone, more tracers than slots, pairs cut by an odd number of slots; and
    from level 6 on short columns' two tracers in the halves of a wavefront, with depths to
    either side of the line."""
    import torch
    from fesom_jax_amd.adjoint import advect_fct_vjp
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh
    from fesom_jax_amd.tracer_adv import FctPlan
    m = icosahedral_mesh(level, nl, seed=111, degree8=degree8)
    c = sharp_case(m, make_case(m, seed=112, dt=2700.0), 1.5)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev)
    Ts = [t(c["T"][0] * (1.0 + 0.1 * j)) for j in range(K)]
    Tos = [t(c["T_old"][0] + 0.2 * j) for j in range(K)]
    gs = [t(g) for g in _cot(m, K, 113)]
    opts = {}
    if split:
        w_i, Z3d, zb3 = _split(m, c, 114)
        opts = dict(w_i=t(w_i), Z3d=t(Z3d), zbar3=t(zb3))
    flow = [t(c[k]) for k in ("uv", "w_e", "helem", "hnode", "hnode_new")]

    def run(js, slots):
        plan = FctPlan(m, torch_dev, max_tracers=slots)
        return advect_fct_vjp(m, *flow, [Ts[j] for j in js], [Tos[j] for j in js],
                              [gs[j] for j in js], dt=c["dt"], plan=plan, **opts)

    one = run(range(K), 1)
    for slots in (2, 3, 4):
        two = run(range(K), slots)
        for j in range(K):
            assert torch.equal(two[0][j], one[0][j]) and torch.equal(two[1][j], one[1][j]), j
        for i in range(2, len(one)):
            assert torch.equal(two[i], one[i]), i


@pytest.mark.parametrize("level,nl,K,split,flat", [
    (6, 8, 2, False, True), (6, 9, 2, False, False), (6, 12, 1, False, True),
    (6, 13, 1, False, False), (6, 8, 1, True, True), (6, 9, 1, True, False),
    (5, 6, 1, False, False)])
def test_short_columns(level, nl, K, split, flat, torch_dev):
    """On a mesh that fills the chip short columns take the flat kernels, either side of the
    line and on a small mesh: the oracle's cotangents, and the workspace of that form."""
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh
    from fesom_jax_amd.tracer_adv import get_plan
    m = icosahedral_mesh(level, nl, seed=131, min_levels=3)
    c = sharp_case(m, make_case(m, seed=132, dt=2700.0), 1.5)
    Ts = [c["T"][0] * (1.0 + 0.1 * j) for j in range(K)]
    Tos = [c["T_old"][0] + 0.2 * j for j in range(K)]
    opts = {}
    if split:
        w_i, Z3d, zb3 = _split(m, c, 133)
        opts = dict(w_i=w_i, Z3d=Z3d, zbar3=zb3)
    gs = _cot(m, K, 134)
    plan = get_plan(m, torch_dev)
    before = plan.own_bytes()
    got = _gpu(m, c, Ts, Tos, gs, torch_dev, **opts)
    NL, DL, EL = m.nod2D * nl, m.edge2D * nl, m.elem2D * nl
    # the flat kernels hold 11 edge arrays, the column kernels 6 (with 30 node and 4
    # triangle arrays each)
    assert (plan.own_bytes() - before > 8 * (34 * NL + 8 * DL + 4 * EL)) == flat
    _compare(f"icosa{level} nl{nl}", got, _oracle(m, c, Ts, Tos, gs, **opts))


def test_workspace_of_one_slot(torch_dev):
    """A plan with one tracer slot reverses no two tracers in one launch, and holds one set of
    cotangents (and the three arrays in which odd tracers are summed apart); its results are
    those of a plan with two sets, bit for bit, with and without the split."""
    import torch
    from fesom_jax_amd.adjoint import advect_fct_vjp
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh
    from fesom_jax_amd.tracer_adv import FctPlan
    m = icosahedral_mesh(4, 35, seed=151, degree8=10)
    c = sharp_case(m, make_case(m, seed=152, dt=2700.0), 1.5)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev)
    Ts = [t(c["T"][0] * (1.0 + 0.1 * j)) for j in range(3)]
    Tos = [t(c["T_old"][0] + 0.2 * j) for j in range(3)]
    gs = [t(g) for g in _cot(m, 3, 153)]
    w_i, Z3d, zb3 = _split(m, c, 154)
    flow = [t(c[k]) for k in ("uv", "w_e", "helem", "hnode", "hnode_new")]
    NL, DL, EL = m.nod2D * 35, m.edge2D * 35, m.elem2D * 35
    lists = 24 * m.edge2D + 8 * m.elem2D + 64
    outs = []
    for slots in (1, 2):
        plan = FctPlan(m, torch_dev, max_tracers=slots)
        before = plan.own_bytes()
        out = list(advect_fct_vjp(m, *flow, Ts, Tos, gs, dt=c["dt"], plan=plan))
        grown = plan.own_bytes() - before
        most = 8 * ((17 * NL + 4 * DL + 2 * EL) if slots == 1 else (31 * NL + 6 * DL + 4 * EL))
        assert grown <= most + slots * (lists + 8 * m.edge2D), (slots, grown, most)
        out += advect_fct_vjp(m, *flow, Ts, Tos, gs, dt=c["dt"], plan=plan, w_i=t(w_i), Z3d=t(Z3d),
                              zbar3=t(zb3))
        outs.append([x for o in out for x in (o if isinstance(o, list) else [o])])
    for i, (x, y) in enumerate(zip(*outs)):
        assert torch.equal(x, y), i


@pytest.mark.parametrize("K,split", [(2, False), (3, True)])
def test_backward_of_large_meshes(K, split, torch_dev):
    """Above 131072 nodes every tracer is reversed alone and the uv, w and w_i cotangents of
    all go into one array each: g_T and g_T_old are those of single-tracer calls bit for
    bit, the others their sums. (A sum of K + 3 K terms of the fields' size, in another
    order: well within 1e-12 of the largest.)"""
    import torch
    from fesom_jax_amd.adjoint import advect_fct_vjp
    from fesom_jax_amd.inputs import make_case
    from fesom_jax_amd.meshgen import icosahedral_mesh
    from fesom_jax_amd.tracer_adv import get_plan
    m = icosahedral_mesh(7, 18, seed=171, land_fraction=0.1)
    assert m.nod2D > 131072
    c = sharp_case(m, make_case(m, seed=172, dt=2700.0), 1.5)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(torch_dev)
    Ts = [t(c["T"][0] * (1.0 + 0.1 * j)) for j in range(K)]
    Tos = [t(c["T_old"][0] + 0.2 * j) for j in range(K)]
    gs = [t(g) for g in _cot(m, K, 173)]
    opts = {}
    if split:
        w_i, Z3d, zb3 = _split(m, c, 174)
        opts = dict(w_i=t(w_i), Z3d=t(Z3d), zbar3=t(zb3))
    flow = [t(c[k]) for k in ("uv", "w_e", "helem", "hnode", "hnode_new")]
    run = lambda js: advect_fct_vjp(m, *flow, [Ts[j] for j in js], [Tos[j] for j in js],
                                    [gs[j] for j in js], dt=c["dt"], **opts)
    print(f"[adjoint] N={m.nod2D} K={K} split={split}", flush=True)
    before = get_plan(m, torch_dev).own_bytes()
    both = run(range(K))
    NL, DL, EL = m.nod2D * 18, m.edge2D * 18, m.elem2D * 18
    # the column kernels' one set (15, 3 and 2 arrays, and the split's), not the flat ones'
    assert get_plan(m, torch_dev).own_bytes() - before < 8 * (20 * NL + 5 * DL + 3 * EL)
    alone = [run([j]) for j in range(K)]
    for j in range(K):
        assert torch.equal(both[0][j], alone[j][0][0]) and torch.equal(both[1][j], alone[j][1][0]), j
    for i in range(2, len(both)):
        want = sum(a[i] for a in alone)
        assert (both[i] - want).abs().max() <= 1e-12 * want.abs().max(), i
