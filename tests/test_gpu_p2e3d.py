"""GPU: 3D Laplace P2M and P2L against direct sums of the solid harmonics
(oracle's definitions), at orders on both sides of the kernel's shapes (row
groups of one, two and four waves; 32, 16 and 8 sources a step), one to 33
densities (weights packed in one tile, one and two tiles, a remainder), real
and complex, S and D."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _setup(order, kind, nrhs):
    from pytential_amd.qbx import QBXLayerPotentialSource
    from pytential_amd.surface import ellipsoid
    d = ellipsoid(1, order=2, fine_order=5)
    src = QBXLayerPotentialSource(d, fine_order=5, qbx_order=2, fmm_order=order,
                                  _max_leaf_refine_weight=70)
    geo = src.qbx_fmm_geometry_data((("self", +1),))
    return d, src, geo, src.make_wrangler(geo, "laplace", 0.0, kind, nrhs)


@pytest.mark.parametrize("order,kind,nrhs,cplx",
                         [(1, "S", 1, False), (2, "D", 1, True), (6, "S", 3, True),
                          (8, "S", 33, False), (8, "S", 17, True), (8, "D", 7, False),
                          (10, "D", 2, True), (11, "D", 11, True), (13, "S", 32, False),
                          (17, "S", 9, True), (20, "D", 1, False), (20, "S", 16, True)])
def test_p2m_and_p2l_match_the_oracle(oracle_lib, order, kind, nrhs, cplx):
    import oracle
    d, src, geo, w = _setup(order, kind, nrhs)
    rng = np.random.default_rng(order)
    dens = rng.normal(size=(d.ndofs, nrhs))
    if cplx:
        dens = dens + 1j * rng.normal(size=(d.ndofs, nrhs))
    st, nrm = w.reorder_sources(src.quad_density(torch.as_tensor(dens)),
                                src.dev["quad_weights"],
                                src.dev["quad_normals"] if kind == "D" else None)
    print(f"order={order} {kind} nrhs={nrhs} complex={cplx}", flush=True)
    m = w.expansions_to_dense(w.form_multipoles(st, nrm))
    loc = w.expansions_to_dense(w.form_locals(st, nrm))
    m, loc = (x.reshape(x.shape[0], x.shape[1], nrhs) for x in (m, loc))
    tree, trav = w.tree, w.traversal
    strengths = st.cpu().numpy().reshape(tree.nsources, nrhs)
    pts = tree.sources.cpu().numpy()
    normals = nrm.cpu().numpy() if kind == "D" else None
    cen = tree.box_centers.cpu().numpy()
    s0 = tree.box_source_starts.cpu().numpy()
    cnt = tree.box_source_counts_nonchild.cpu().numpy()
    kp = oracle.kparams("laplace", 0.0, kind, 2, dim=3)

    def direct(idx, box, local):
        return np.stack([oracle.p2e(kp, "laplace", local, order, cen[:, box], 1.0, pts[:, idx],
                                    None if normals is None else normals[:, idx],
                                    strengths[idx, r]) for r in range(nrhs)], axis=-1)
    boxes = trav.source_boxes.cpu().numpy()
    for b in boxes[:: max(1, len(boxes) // 6)]:
        ref = direct(np.arange(s0[b], s0[b] + cnt[b]), b, 0)
        assert np.max(np.abs(m[b] - ref)) < 1e-12 * np.max(np.abs(ref))
    starts = trav.from_sep_bigger_starts.cpu().numpy()
    lists = trav.from_sep_bigger_lists.cpu().numpy()
    ttp = trav.target_or_target_parent_boxes.cpu().numpy()
    full = np.nonzero(np.diff(starts))[0]
    assert len(full) > 0
    for i in full[:: max(1, len(full) // 6)]:
        idx = np.concatenate([np.arange(s0[b], s0[b] + cnt[b])
                              for b in lists[starts[i]:starts[i + 1]]])
        ref = direct(idx, ttp[i], 1)
        n = np.floor(np.sqrt(np.arange((order + 1) ** 2))).astype(int)
        # each degree against its own size: the coefficients grow like r^-n
        for deg in range(order + 1):
            sel = n == deg
            assert np.max(np.abs(loc[ttp[i]][sel] - ref[sel])) < 1e-12 * np.max(np.abs(ref[sel]))
