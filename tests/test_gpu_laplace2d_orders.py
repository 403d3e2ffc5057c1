"""GPU: 2D Laplace expansions against the oracle's at the orders where the
kernels change shape (16, 32 and 64 lanes to a box's coefficients, the last
order their LDS holds and the first beyond it), with orders that differ
between levels, S and D, one and several densities (a chunk of four and of
eight and remainders)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _rel(a, b):
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("orders,kind,nrhs", [((1,), "S", 1), ((15,), "D", 3), ((16,), "S", 9),
                                              ((31,), "S", 1), ((32, 20), "D", 2),
                                              ((40, 7), "S", 5), ((41,), "D", 1)])
def test_stages_match_the_oracle(oracle_lib, orders, kind, nrhs):
    import oracle

    from pytential_amd import problems
    from pytential_amd.qbx import QBXLayerPotentialSource
    cfg = problems.refine_until_associated(problems.config1(nelements=48, grid_n=40),
                                           oracle.assoc_status_and_flags)
    d = cfg.discr
    src = QBXLayerPotentialSource(
        d, fine_order=d.fine_order, qbx_order=3, _max_leaf_refine_weight=24,
        fmm_level_to_order=lambda k, a, tree, lev: orders[min(lev, len(orders) - 1)]
        if lev < 3 else orders[-1])
    geo = src.qbx_fmm_geometry_data(((cfg.targets, cfg.target_sides),))
    ref = oracle.GeometryData(d, cfg.targets, cfg.target_sides, max_leaf_refine_weight=24)
    assert len(ref.trav.from_sep_bigger_lists) > 0
    w = src.make_wrangler(geo, "laplace", 0.0, kind, nrhs)
    lo = list(w._lo)
    print(f"orders={lo} {kind} nrhs={nrhs}", flush=True)
    rng = np.random.default_rng(3)
    dens = rng.normal(size=(d.ndofs, nrhs))
    st, nrm = w.reorder_sources(src.quad_density(dens if nrhs > 1 else dens[:, 0]),
                                src.dev["quad_weights"],
                                src.dev["quad_normals"] if kind == "D" else None)
    m = w.coarsen_multipoles(w.form_multipoles(st, nrm))
    loc = w.multipole_to_local(m)
    w.refine_locals(w.form_locals(st, nrm, loc))
    m, loc = (w.expansions_to_dense(x) for x in (m, loc))
    m, loc = (x.reshape(x.shape[0], x.shape[1], nrhs) for x in (m, loc))
    q = w.form_global_qbx_locals(st, nrm).cpu().numpy().reshape(geo.ncenters, -1, nrhs)
    assert np.isfinite(q).all()
    for r in range(nrhs):
        _, stg = ref.fmm("laplace", 0.0, kind, 3, lo, d.strengths(dens[:, r]),
                         return_stages=True)
        # the repository's bound for stages on the same tree
        assert _rel(m[:, :, r], stg["mpole"]) < 1e-12
        assert _rel(loc[:, :, r], stg["local"]) < 1e-12
