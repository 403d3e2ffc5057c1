"""GPU: adjoint drivers that meet in time keep apart: one captured into a HIP
graph while another context's runs eagerly on a stream of its own, and both
again between replays.  Against the eager results; each stage adds by atomics,
so to the rounding of its sums."""
import ctypes as ct

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

np = pytest.importorskip("numpy")


def _adjoint(w, pot_adj, nrm, out, stream):
    from pytential_amd import _lib
    from pytential_amd import fmm as F
    _lib.call("qbx_drive_fmm_adjoint", w.ctx.h, stream.cuda_stream, w.tree.h, w.traversal.h,
              w.geo.h, ct.byref(w.kd), F._p(pot_adj), F._p(nrm), F._p(out))


@pytest.mark.parametrize("kernel,k", [("laplace", 0.0), ("helmholtz", 8.0)])
def test_capture_beside_an_eager_call(kernel, k):
    from test_gpu_adjoint2d import _rnd, _setup
    sides = []
    for i in range(2):
        d, src, pairs = _setup(kernel, k, "S")
        w = src.make_wrangler(src.qbx_fmm_geometry_data(tuple(pairs)), kernel, k, "S", 1,
                              private_context=True)
        ya = _rnd(w.full_output_zeros().numel(), np.random.default_rng(i),
                  real=kernel == "laplace")
        out = torch.zeros(w.tree.nsources, dtype=torch.complex128, device="cuda")
        s = torch.cuda.Stream()
        _adjoint(w, ya, None, out, torch.cuda.current_stream())
        torch.cuda.synchronize()
        sides.append((w, ya, out, s, out.clone()))
    (wa, ya, oa, sa, ra), (wb, yb, ob, sb, rb) = sides
    assert wa.ctx.h.value != wb.ctx.h.value

    def close(x, r):
        return float((x - r).abs().max()) < 1e-12 * float(r.abs().max())
    oa.zero_()
    ob.zero_()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=sa, capture_error_mode="relaxed"):
        _adjoint(wa, ya, None, oa, sa)
        _adjoint(wb, yb, None, ob, sb)
    torch.cuda.synchronize()
    assert float(oa.abs().max()) == 0.0 and close(ob, rb)
    for _ in range(4):
        oa.zero_()
        ob.zero_()
        g.replay()
        torch.cuda.synchronize()
        print(f"[replay] {kernel}", flush=True)
        assert close(oa, ra) and float(ob.abs().max()) == 0.0
        for w, y, o, s, r in sides:
            o.zero_()
            torch.cuda.synchronize()
            _adjoint(w, y, None, o, s)
            s.synchronize()
            assert close(o, r)
