"""GPU: the transposed stages where the expansion orders differ between levels
(rising, falling, and up to the largest), level by level.

Each stage against its forward stage through Re <y', A x> = Re <A^H y', x>, x
what the forward's earlier stages make of random strengths and y' what the
transposed later stages make of random potential adjoints, so that every level
counts; then with y' (or, where the expansions are the input, x) of one level
alone.  Both sides round sums of up to a few thousand products, which at 2^-53
each and at random leave 1e-14 of sum |y'_i| |(A x)_i|: 1e-13.
"""
import functools

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

np = pytest.importorskip("numpy")

FALLING = (120, 120, 120, 60, 30, 15, 12, 10, 8)


def _dot(a, b):
    return float(torch.sum(torch.conj(a.reshape(-1)) * b.reshape(-1)).real)


def _wrangler2d(kernel, k, kind, orders):
    from test_gpu_adjoint2d import _config

    from pytential_amd.qbx import QBXLayerPotentialSource
    cfg = _config()
    d = cfg.discr
    src = QBXLayerPotentialSource(d, fine_order=d.fine_order, qbx_order=4,
                                  fmm_level_to_order=lambda kn, a, t, lev:
                                  orders[lev % len(orders)])
    pairs = (("self", +1), (cfg.targets[:, d.ndofs:], 0))
    return src, src.make_wrangler(src.qbx_fmm_geometry_data(pairs), kernel, k, kind, 1)


@functools.lru_cache(maxsize=1)
def _sphere():
    from pytential_amd.surface import icosphere
    rng = np.random.default_rng(5)
    v = rng.normal(size=(3, 400))
    v /= np.linalg.norm(v, axis=0)
    return icosphere(2, order=4, fine_order=5), v * rng.uniform(1.2, 3.0, 400)


def _wrangler3d(k, orders):
    from pytential_amd.qbx import QBXLayerPotentialSource
    d, tgt = _sphere()
    src = QBXLayerPotentialSource(d, fine_order=d.fine_order, qbx_order=3,
                                  fmm_level_to_order=lambda kn, a, t, lev:
                                  orders[lev % len(orders)], _max_leaf_refine_weight=64)
    return src, src.make_wrangler(src.qbx_fmm_geometry_data((("self", +1), (tgt, 0))),
                                  "helmholtz", k, "S", 1)


@pytest.mark.parametrize("dim,kernel,k,kind,orders", [
    (2, "laplace", 0.0, "S", (31, 12, 45, 5)),
    (2, "laplace", 0.0, "D", (5, 31, 12, 20)),
    (2, "helmholtz", 40.0, "S", (31, 12, 70, 5)),
    (2, "helmholtz", 40.0, "D", (5, 70, 12, 31)),
    (2, "helmholtz", 60.0, "D", FALLING),
    (2, "helmholtz", 200.0, "S", (40, 40, 40, 70, 120, 120, 50, 30)),
    (3, "helmholtz", 1.7, "S", (10, 7, 12, 4)),
    (3, "helmholtz", 1.7, "S", (13, 4, 9, 12, 3, 10))])
def test_stages_level_by_level(dim, kernel, k, kind, orders):
    from pytential_amd import fmm as F
    src, w = _wrangler2d(kernel, k, kind, orders) if dim == 2 else _wrangler3d(k, orders)
    rng = np.random.default_rng(11)
    ns, npot = w.tree.nsources, w.full_output_zeros().numel()
    real = kernel == "laplace"

    def rnd(n):
        x = rng.normal(size=n) + (0.0 if real else 1j * rng.normal(size=n))
        return torch.as_tensor(x, dtype=torch.complex128, device="cuda")
    q, yp = rnd(ns), rnd(npot)
    nrm = w.reorder_sources(torch.zeros(ns, dtype=torch.complex128, device="cuda"),
                            src.dev["quad_weights"],
                            src.dev["quad_normals"])[1] if kind == "D" else None

    def adj(stage, y):
        return F.adjoint_stage(w, stage, y.clone(), normals=nrm)
    # the forward's arrays and the adjoint's
    m0 = w.form_multipoles(q, nrm)
    m = w.coarsen_multipoles(m0.clone())
    l0 = w.multipole_to_local(m) + w.form_locals(q, nrm)
    loc = w.refine_locals(l0.clone())
    qe = w.form_global_qbx_locals(q, nrm).reshape(-1)
    yq = adj("eval_qbx_expansions", yp).reshape(-1)
    yl = adj("eval_locals", yp) + adj("translate_box_local_to_qbx_local", yq)
    yl0 = adj("refine_locals", yl)
    ym = (adj("multipole_to_local", yl0) + adj("eval_multipoles", yp)
          + adj("translate_box_multipoles_to_qbx_local", yq))
    ym0 = adj("coarsen_multipoles", ym)
    OUT, IN = "out", "in"
    stages = [
        ("form_multipoles", lambda x: w.form_multipoles(x, nrm), q, ym0, OUT),
        ("coarsen_multipoles", lambda x: w.coarsen_multipoles(x.clone()), m0, ym, OUT),
        ("eval_direct", lambda x: w.eval_direct(x, nrm), q, yp, None),
        ("multipole_to_local", w.multipole_to_local, m, yl0, OUT),
        ("eval_multipoles", w.eval_multipoles, m, yp, IN),
        ("form_locals", lambda x: w.form_locals(x, nrm), q, yl0, OUT),
        ("refine_locals", lambda x: w.refine_locals(x.clone()), l0, yl, OUT),
        ("eval_locals", w.eval_locals, loc, yp, IN),
        ("form_global_qbx_locals", lambda x: w.form_global_qbx_locals(x, nrm), q, yq, None),
        ("translate_box_multipoles_to_qbx_local", w.translate_box_multipoles_to_qbx_local, m, yq,
         IN),
        ("translate_box_local_to_qbx_local", w.translate_box_local_to_qbx_local, loc, yq, IN),
        ("eval_qbx_expansions", w.eval_qbx_expansions, qe, yp, None),
    ]
    off = w.level_offsets

    def level(x, lev):
        y = torch.zeros_like(x)
        y[off[lev]:off[lev + 1]] = x[off[lev]:off[lev + 1]]
        return y
    for name, f, x, y, side in stages:
        seen, worst = [], 0.0
        for lev in [None] + list(range(w.tree.nlevels) if side else ()):
            xv = level(x, lev) if lev is not None and side == IN else x
            yv = level(y, lev) if lev is not None and side == OUT else y
            ax = f(xv).reshape(-1)
            scale = float(torch.sum(yv.reshape(-1).abs() * ax.abs()))
            if scale == 0.0:
                assert lev is not None, name    # no stage may be empty
                continue
            xa = adj(name, yv).reshape(-1)
            err = abs(_dot(yv, ax) - _dot(xa, xv)) / scale
            worst = max(worst, err)
            seen.append(lev)
            assert err < 1e-13, (name, lev, err)
        print(f"[adjoint] {dim}D {kernel} {kind} {orders[:4]} {name}: levels {seen[1:]} "
              f"{worst:.1e}", flush=True)
        assert side is None or len(seen) > 1, name
