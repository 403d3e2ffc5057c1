"""GPU: 3D Helmholtz QBX expansions (P2QBXL + M2QBXL + L2QBXL) against the
oracle at the QBX orders the register kernel is built for and the first
beyond, S and D, on a tree of small leaves: list 1 of the coarse boxes holds
more than one tile of 256 entries, and the target boxes hold one, two and more
centers (one, two or four waves a center), two densities launched in turn."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("pq,kind,leaf", [(0, "S", 16), (1, "D", 6), (2, "S", 6), (3, "S", 6),
                                          (3, "D", 16), (4, "S", 16), (5, "S", 6), (5, "D", 16),
                                          (6, "S", 16)])
def test_qbx_expansions_match_oracle(oracle_lib, pq, kind, leaf):
    import oracle

    from pytential_amd.qbx import QBXLayerPotentialSource
    from pytential_amd.surface import ellipsoid
    d = ellipsoid(1, order=3, fine_order=5)
    src = QBXLayerPotentialSource(d, fine_order=5, qbx_order=pq, fmm_order=4,
                                  _max_leaf_refine_weight=leaf)
    geo = src.qbx_fmm_geometry_data((("self", +1),))
    ref = oracle.GeometryData(d, d.nodes, np.ones(d.ndofs, np.int32),
                              max_leaf_refine_weight=leaf)
    n1 = np.diff(ref.trav.neighbor_source_boxes_starts)
    per = np.bincount(geo.qbx_center_to_target_box().cpu().numpy())
    print(f"pq={pq} {kind} leaf={leaf}: lists up to {n1.max()}, centers a box {set(per)}",
          flush=True)
    assert n1.max() > 256 or leaf > 6
    rng = np.random.default_rng(pq)
    dens = rng.normal(size=(d.ndofs, 2)) + 1j * rng.normal(size=(d.ndofs, 2))
    w = src.make_wrangler(geo, "helmholtz", 5.0, kind, nrhs=2)
    st, nrm = w.reorder_sources(src.quad_density(torch.as_tensor(dens)),
                                src.dev["quad_weights"],
                                src.dev["quad_normals"] if kind == "D" else None)
    m = w.coarsen_multipoles(w.form_multipoles(st, nrm))
    loc = w.multipole_to_local(m)
    w.refine_locals(w.form_locals(st, nrm, loc))
    q = w.form_global_qbx_locals(st, nrm)
    w.translate_box_multipoles_to_qbx_local(m, q)
    w.translate_box_local_to_qbx_local(loc, q)
    q = q.cpu().numpy()
    for r in range(2):
        _, stages = ref.fmm("helmholtz", 5.0, kind, pq, [4] * ref.tree.nlevels,
                            d.strengths(dens[:, r]), return_stages=True)
        # the repository's bound for stages on the same tree
        assert np.max(np.abs(q[:, :, r] - stages["qbx"])) < 1e-12 * np.max(np.abs(stages["qbx"]))
