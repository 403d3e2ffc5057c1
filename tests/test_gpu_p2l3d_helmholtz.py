"""GPU: P2L of 3D Helmholtz at every order of the register kernel, the first
beyond it, and per-level orders that change inside it, against the oracle's
expansions of the list-4 sources.  Some boxes' lists hold more than one chunk of
256 sources; two densities are launched in turn."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

K = 5.0


@pytest.mark.parametrize("orders,kind", [(o, "S") for o in range(1, 14)] +
                         [("mixed", "S"), (4, "D")])
def test_locals_match_oracle(oracle_lib, orders, kind):
    import oracle

    from pytential_amd.qbx import QBXLayerPotentialSource
    from pytential_amd.surface import ellipsoid
    d = ellipsoid(2, order=3, fine_order=5)
    rng = np.random.default_rng(7)
    # loose targets: coarse leaves beside the surface's small ones, so list 4
    loose = rng.normal(size=(3, 200))
    loose *= rng.uniform(2.0, 3.5, 200) / np.linalg.norm(loose, axis=0)

    def level_to_order(kernel, kernel_args, tree, level):
        return (3, 9, 5, 12, 7, 13)[level % 6] if orders == "mixed" else orders

    src = QBXLayerPotentialSource(d, fine_order=5, qbx_order=2,
                                  fmm_level_to_order=level_to_order,
                                  _max_leaf_refine_weight=64)
    geo = src.qbx_fmm_geometry_data((("self", +1), (loose, 0)))
    dens = rng.normal(size=(d.ndofs, 2)) + 1j * rng.normal(size=(d.ndofs, 2))
    w = src.make_wrangler(geo, "helmholtz", K, kind, nrhs=2)
    st, nrm = w.reorder_sources(src.quad_density(torch.as_tensor(dens)),
                                src.dev["quad_weights"],
                                src.dev["quad_normals"] if kind == "D" else None)
    loc = w.expansions_to_dense(w.form_locals(st, nrm))
    tree, trav = w.tree, w.traversal
    strengths, pts = st.cpu().numpy().reshape(tree.nsources, 2), tree.sources.cpu().numpy()
    normals = nrm.cpu().numpy() if kind == "D" else None
    cen = tree.box_centers.cpu().numpy()
    s0 = tree.box_source_starts.cpu().numpy()
    cnt = tree.box_source_counts_nonchild.cpu().numpy()
    level = tree.box_levels.cpu().numpy()
    starts = trav.from_sep_bigger_starts.cpu().numpy()
    lists = trav.from_sep_bigger_lists.cpu().numpy()
    ttp = trav.target_or_target_parent_boxes.cpu().numpy()
    kp = oracle.kparams("helmholtz", K, kind, 2, dim=3)
    full = np.nonzero(np.diff(starts))[0]
    seen = set()
    most = 0
    for i in full[:: max(1, len(full) // 24)]:
        b = ttp[i]
        p = level_to_order(None, None, None, level[b])
        idx = np.concatenate([np.arange(s0[e], s0[e] + cnt[e])
                              for e in lists[starts[i]:starts[i + 1]]])
        if len(idx) == 0:
            continue
        seen.add(p)
        most = max(most, len(idx))
        n = np.floor(np.sqrt(np.arange((p + 1) ** 2))).astype(int)
        scale = min(1.0, K * tree.root_extent * 2.0 ** -level[b]) ** n
        for r in range(2):
            ref = scale * oracle.p2e(kp, "helmholtz", 1, p, cen[:, b], 1.0, pts[:, idx],
                                     None if normals is None else normals[:, idx],
                                     strengths[idx, r])
            # each degree against its own size: a few hundred rounded products
            for deg in range(p + 1):
                err = np.abs(loc[b, :len(n), r] - ref)[n == deg].max()
                assert err < 1e-12 * np.abs(ref[n == deg]).max(), (p, deg, err)
    print(f"orders {sorted(seen)} {kind}: {len(full)} boxes, up to {most} sources", flush=True)
    assert most > 256 and (orders != "mixed" or len(seen) > 1)
