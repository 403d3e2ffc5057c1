"""GPU: the tree's box weights and the traversal's lists where their kernels
change branches, bit-exact against the CPU oracle on random points.

* list lengths around the rank sort's 256 entries and far above (targets with
  a large extent stop in coarse boxes and list thousands of leaves);
* more boxes than one window of the sort's bitmap holds (262144);
* levels of more than 2048 boxes (weights straight to global memory) and of
  fewer (summed in LDS first), particles in an order with runs of equal boxes
  and without, weights above one.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# dim, sources, leaf weight, targets, target radius, list-3 threshold, sorted input
CASES = [(2, 1, 1, 1, 0.0, 15, False), (2, 300, 1, 40, 0.2, 0, False),
         (2, 5000, 8, 700, 0.3, 15, True), (3, 4000, 4, 300, 0.25, 30, False),
         (3, 60000, 16, 20, 0.4, 0, True), (2, 300000, 3, 12, 0.35, 3, False)]


@pytest.mark.parametrize("dim,ns,leaf,nt,rad,mins,ordered", CASES)
def test_tree_and_lists_bit_exact(oracle_lib, dim, ns, leaf, nt, rad, mins, ordered):
    import oracle

    from pytential_amd.geometry import Traversal, Tree
    from test_gpu_parity import TRAV_FIELDS, TREE_FIELDS
    rng = np.random.default_rng(17 + ns)
    src = rng.uniform(-1, 1, (dim, ns))
    src[:, :ns // 4] *= 0.01                      # a dense corner: deep levels
    if ordered:
        src = src[:, np.argsort(src[0])]
    tgt = rng.uniform(-1, 1, (dim, nt))
    radii = np.where(np.arange(nt) % 3 == 0, rad, 0.01 * rad)
    sw = rng.integers(1, 4, ns).astype(np.int32)
    tw = rng.integers(0, 3, nt).astype(np.int32)
    print(f"dim={dim} ns={ns} leaf={leaf} nt={nt}", flush=True)
    t = Tree(src, tgt, radii, sw, tw, leaf)
    r = oracle.Tree(src, tgt, radii, sw, tw, max_leaf_refine_weight=leaf)
    for f in TREE_FIELDS:
        assert np.array_equal(getattr(t, f).cpu().numpy(), getattr(r, f)), f
    tr = Traversal(t, 2, True, mins)
    rr = oracle.Traversal(r, 2, True, mins)
    for f in TRAV_FIELDS:
        assert np.array_equal(getattr(tr, f).cpu().numpy(), getattr(rr, f)), f
    if ns == 300000:
        assert t.nboxes > 262144
        n1 = np.diff(rr.neighbor_source_boxes_starts)
        assert n1.max() > 256
