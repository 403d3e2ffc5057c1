"""GPU: the 3D Helmholtz point sums and their adjoint against torch's FP64
dense sums, at the sizes where the kernels change shape: one point, tile
remainders, and source counts on both sides of the adjoint's 16, 4 and 1
threads a source; with coincident points (zero) and with phases beyond the
reduced range of the sine (1.6e6), whose tiles are summed a second time."""
import ctypes as ct
import math

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _p(t):
    return ct.c_void_p(t.data_ptr())


@pytest.mark.parametrize("ns,nt,k", [(1, 1, 2.0), (300, 257, 5.0), (65535, 40, 5.0),
                                     (65536, 300, 0.7), (262143, 33, 3.0), (262400, 257, 5.0),
                                     (700, 300, 1.3e6)])
def test_far_sums_and_adjoint(ns, nt, k):
    from pytential_amd._lib import call
    from pytential_amd.geometry import Context, _stream
    gen = torch.Generator(device="cuda").manual_seed(ns + nt)
    f64 = dict(dtype=torch.float64, device="cuda", generator=gen)
    src, tgt = torch.randn((3, ns), **f64), 2 * torch.randn((3, nt), **f64)
    if ns > 100:
        tgt[:, nt // 2] = src[:, 77]              # coincident: contributes zero
    q = torch.complex(torch.randn(ns, **f64), torch.randn(ns, **f64))
    u = torch.complex(torch.randn(nt, **f64), torch.randn(nt, **f64))
    print(f"ns={ns} nt={nt} k={k}", flush=True)
    pot, dk = torch.empty_like(u), torch.empty_like(u)
    v = torch.empty_like(q)
    h = Context.get().h
    call("qbx_helmholtz3d_p2p", h, _stream(), ns, _p(src), _p(q), nt, _p(tgt), k, _p(pot),
         _p(dk))
    call("qbx_helmholtz3d_p2p_adjoint", h, _stream(), ns, _p(src), nt, _p(tgt), k, _p(u), _p(v))
    ref = [torch.zeros_like(u), torch.zeros_like(u), torch.zeros_like(q)]
    size = [torch.zeros(nt, dtype=torch.float64, device="cuda"),
            torch.zeros(nt, dtype=torch.float64, device="cuda"),
            torch.zeros(ns, dtype=torch.float64, device="cuda")]
    for a in range(0, nt, 16):
        d = tgt[:, a:a + 16, None] - src[:, None, :]
        r = torch.sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2])
        on = r > 0
        e = torch.polar(on.to(torch.float64), k * r) / (4 * math.pi)
        g = e / torch.where(on, r, 1.0)
        # the phase k r carries its own rounding
        w = on * (1 + k * r) / (4 * math.pi)
        ref[0][a:a + 16], ref[1][a:a + 16] = g @ q, 1j * (e @ q)
        ref[2] += (u[a:a + 16].conj() @ g).conj()
        size[0][a:a + 16] = (w / torch.where(on, r, 1.0)) @ q.abs()
        size[1][a:a + 16] = w @ q.abs()
        size[2] += u[a:a + 16].abs() @ (w / torch.where(on, r, 1.0))
    # 16 roundings of each term (r, the phase, sine and cosine, products) and
    # the sums' own, against the terms' absolute values
    for got, want, bound in zip((pot, dk, v), ref, size):
        assert bool(((got - want).abs() <= 16 * 2.3e-16 * bound).all())
