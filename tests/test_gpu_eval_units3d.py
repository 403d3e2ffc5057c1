"""GPU: 3D Laplace P2P and M2P over the geometry's work units against the
oracle's QBX-FMM, at loose points whose boxes hold one, a few and more than 64
of them, near and far from the surface, S and D, one and several densities
(1, 8 and 9 columns: a full chunk of right-hand sides and a remainder)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("kind,npoints,nrhs", [("S", 1, 1), ("D", 63, 1), ("D", 700, 9),
                                               ("S", 2000, 8)])
def test_loose_points_match_oracle(oracle_lib, kind, npoints, nrhs):
    import oracle

    from pytential_amd import surface
    from pytential_amd.qbx import QBXLayerPotentialSource
    d = surface.ellipsoid(2, order=2, fine_order=4)
    rng = np.random.default_rng(5)
    pts = rng.normal(size=(3, npoints))
    pts *= rng.uniform(1.3, 4.0, npoints) / np.linalg.norm(pts, axis=0)
    pts[:, npoints // 2:] = pts[:, :1] + 1e-3 * rng.normal(size=(3, npoints - npoints // 2))
    dens = rng.normal(size=(d.ndofs, nrhs))
    src = QBXLayerPotentialSource(d, fine_order=4, qbx_order=2, fmm_order=6)
    pot, = src.exec_compute_potential("laplace", torch.as_tensor(dens, device="cuda"),
                                      [(pts, 0)], source_kind=kind)
    pot = pot.cpu().numpy().reshape(npoints, nrhs)
    g = oracle.GeometryData(d, pts, np.zeros(npoints, np.int32), max_leaf_refine_weight=512,
                            from_sep_smaller_min_nsources_cumul=30)
    for r in range(nrhs):
        ref, _ = g.fmm("laplace", 0.0, kind, 2, [6] * g.tree.nlevels, d.strengths(dens[:, r]))
        # the repository's bound for potentials on the same tree
        assert np.max(np.abs(pot[:, r] - ref.real)) < 1e-12 * np.max(np.abs(ref))
