"""GPU: the transposed 2D Helmholtz stages at the edges of their batches.

The kernels size their batches of points by the expansion order and the LDS of
a block, and split a block's threads into slices by the number of
coefficients: orders 1 (most slices, full batches), 31 (2 p + 1 = 63, one below
a wavefront), 32 and 70 (batches of a few points).  Each stage against its
forward stage through Re <y', A x> = Re <A^H y', x> on random inputs; both
sides round sums of a few thousand products, so 1e-12 (4500 ulp) of
|y'| |A x|.  And the whole chain on one stream against the default.
"""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

np = pytest.importorskip("numpy")


def _wrangler(kind, fmm_order, k=40.0):
    from test_gpu_adjoint2d import _setup
    d, src, pairs = _setup("helmholtz", k, kind, fmm_order)
    w = src.make_wrangler(src.qbx_fmm_geometry_data(tuple(pairs)), "helmholtz", k, kind, 1)
    ns = w.tree.nsources
    _, nrm = w.reorder_sources(torch.zeros(ns, dtype=torch.complex128, device="cuda"),
                               src.dev["quad_weights"],
                               src.dev["quad_normals"] if kind == "D" else None)
    return w, nrm


@pytest.mark.parametrize("kind", ["S", "D"])
@pytest.mark.parametrize("order", [1, 31, 32, 70])
def test_stages_at_order(order, kind):
    from test_gpu_adjoint2d import _dot, _rnd

    from pytential_amd import fmm as F
    w, nrm = _wrangler(kind, order)
    rng = np.random.default_rng(order)
    ns, nm = w.tree.nsources, w.multipole_expansion_zeros().numel()
    nq, npot = w.qbx_local_expansion_zeros().numel(), w.full_output_zeros().numel()
    fw = {
        "form_multipoles": (lambda x: w.form_multipoles(x, nrm), ns, nm),
        "coarsen_multipoles": (lambda x: w.coarsen_multipoles(x.clone()), nm, nm),
        "eval_direct": (lambda x: w.eval_direct(x, nrm), ns, npot),
        "multipole_to_local": (lambda x: w.multipole_to_local(x), nm, nm),
        "eval_multipoles": (lambda x: w.eval_multipoles(x), nm, npot),
        "form_locals": (lambda x: w.form_locals(x, nrm), ns, nm),
        "refine_locals": (lambda x: w.refine_locals(x.clone()), nm, nm),
        "eval_locals": (lambda x: w.eval_locals(x), nm, npot),
        "form_global_qbx_locals": (lambda x: w.form_global_qbx_locals(x, nrm), ns, nq),
        "translate_box_multipoles_to_qbx_local":
            (lambda x: w.translate_box_multipoles_to_qbx_local(x), nm, nq),
        "translate_box_local_to_qbx_local":
            (lambda x: w.translate_box_local_to_qbx_local(x), nm, nq),
        "eval_qbx_expansions": (lambda x: w.eval_qbx_expansions(x), nq, npot),
    }
    for stage, (f, nin, nout) in fw.items():
        x, ya = _rnd(nin, rng), _rnd(nout, rng)
        y = f(x).reshape(-1)
        xa = F.adjoint_stage(w, stage, ya.clone(), normals=nrm).reshape(-1)
        scale = float(torch.linalg.norm(ya) * torch.linalg.norm(y)) + 1e-300
        assert float(torch.linalg.norm(y)) > 0, stage
        err = abs(_dot(ya, y).real - _dot(xa, x).real) / scale
        print(f"[adjoint] order {order} {kind} {stage}: {err:.1e}", flush=True)
        assert err < 1e-12, (stage, err)


@pytest.mark.parametrize("kernel,k", [("laplace", 0.0), ("helmholtz", 8.0)])
def test_chain_on_one_stream(kernel, k):
    from test_gpu_adjoint2d import _rnd, _setup

    from pytential_amd import _lib
    from pytential_amd import fmm as F
    d, src, pairs = _setup(kernel, k, "S")
    w = src.make_wrangler(src.qbx_fmm_geometry_data(tuple(pairs)), kernel, k, "S", 1)
    n = w.full_output_zeros().numel()
    y = F.drive_fmm_fused(w, torch.ones(w.tree.nsources, dtype=torch.complex128, device="cuda"),
                          None)
    ya = _rnd(y.numel(), np.random.default_rng(n), real=kernel == "laplace")
    many = [F.drive_fmm_adjoint(w, ya, None) for _ in range(3)]
    _lib.call("qbx_ctx_set_tuning", w.ctx.h, _lib.TUNE_DRIVE_STREAMS, 1)
    try:
        one = F.drive_fmm_adjoint(w, ya, None)
    finally:
        _lib.call("qbx_ctx_set_tuning", w.ctx.h, _lib.TUNE_DRIVE_STREAMS, 4)
    scale = float(one.abs().max())
    for m in many:
        assert float((m - one).abs().max()) < 1e-12 * scale
