"""GPU: 3D Helmholtz M2QBXL of one density, whose waves come from tables, and its
transpose, from the lowest to the largest sum of box and QBX order (20 + 3).
Forward: against the same stage of two densities, another kernel with its own
recurrences (checked against the oracle elsewhere), each QBX order n against its
own size, 1e-12 (a few thousand rounded products).  Transpose: Re <y', A x> = Re
<A^H y', x> to 1e-12 of |y'| |A x|, the bound of the other adjoint tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("p,pq", [(1, 0), (2, 1), (7, 2), (10, 3), (20, 3)])
def test_m2qbxl_and_transpose(p, pq):
    from pytential_amd import fmm as F
    from pytential_amd.qbx import QBXLayerPotentialSource
    from pytential_amd.surface import ellipsoid
    d = ellipsoid(2, order=3, fine_order=5)
    src = QBXLayerPotentialSource(d, fine_order=5, qbx_order=pq, fmm_order=p,
                                  _max_leaf_refine_weight=64)
    geo = src.qbx_fmm_geometry_data((("self", +1),))
    assert len(geo.traversal().from_sep_smaller_lists) > 0
    rng = np.random.default_rng(p)
    dens = rng.normal(size=(d.ndofs, 2)) + 1j * rng.normal(size=(d.ndofs, 2))
    q = []
    for nrhs in (1, 2):
        w = src.make_wrangler(geo, "helmholtz", 5.0, "S", nrhs)
        st, _ = w.reorder_sources(
            src.quad_density(torch.as_tensor(dens if nrhs == 2 else dens[:, 0].copy())),
            src.dev["quad_weights"], None)
        m = w.coarsen_multipoles(w.form_multipoles(st, None))
        q.append(w.translate_box_multipoles_to_qbx_local(m))
        if nrhs == 1:
            one, m1 = w, m
    got = q[0].reshape(-1, (pq + 1) ** 2)
    ref = q[1].reshape(-1, (pq + 1) ** 2, 2)[:, :, 0]
    for n in range(pq + 1):
        s = slice(n * n, (n + 1) ** 2)
        scale = float(ref[:, s].abs().max())
        assert scale > 0 and float((got - ref)[:, s].abs().max()) < 1e-12 * scale, n
    x = torch.as_tensor(rng.normal(size=m1.numel()) + 1j * rng.normal(size=m1.numel()),
                        device="cuda")
    y = one.translate_box_multipoles_to_qbx_local(x).reshape(-1)
    ya = torch.as_tensor(rng.normal(size=y.numel()) + 1j * rng.normal(size=y.numel()),
                         device="cuda")
    xa = F.adjoint_stage(one, "translate_box_multipoles_to_qbx_local", ya.clone()).reshape(-1)
    lhs = complex(torch.sum(torch.conj(ya) * y)).real
    rhs = complex(torch.sum(torch.conj(xa) * x)).real
    scale = float(torch.linalg.norm(ya) * torch.linalg.norm(y))
    print(f"p={p} pq={pq}: transpose {abs(lhs - rhs) / scale:.1e}", flush=True)
    assert abs(lhs - rhs) < 1e-12 * scale
