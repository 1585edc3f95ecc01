"""Vocabulary-tree descent at the sizes where the score and the exact kernels can go wrong:
branch counts around the 32-child blocks and the 64-child steps, slots with one key and with
31 absent ones, keys and trees of other scales (the scores are formed on scaled FP16 parts),
and scales outside the certified range.  The leaves are whole numbers: they equal the
oracle's."""
import numpy as np
import pytest

from oracle import oracle
from v3dmatch import voctree

pytestmark = pytest.mark.gpu


def _case(branch, depth, n, seed):
    rng = np.random.default_rng(seed)
    n_nodes, _ = voctree.sizes(branch, depth)
    tree = rng.standard_normal((n_nodes, 128)).astype(np.float32)
    tree /= np.linalg.norm(tree, axis=1, keepdims=True)
    if branch > 2:
        tree[branch - 1] = tree[1]                      # an exact tie with the last child
    keys = tree[rng.integers(0, n_nodes, n)] + 0.05 * rng.standard_normal((n, 128))
    return tree, keys.astype(np.float32)


def _same(tree, branch, depth, keys):
    with voctree.VocabularyTree(branch, depth) as t:
        t.setNodes(tree)
        got = t.traverseTree(keys.shape[0], keys)
        exact = t.synchronize()
    want = oracle.voctree_leaves(tree, branch, depth, keys, global_ids=True)
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, (bad[:8], got[bad[:8]], want[bad[:8]])
    return exact


@pytest.mark.parametrize("branch,depth", [(2, 6), (31, 2), (32, 2), (33, 2), (63, 2), (64, 2), (65, 2), (128, 2),
                                          (257, 1)])
@pytest.mark.parametrize("n", [1, 127, 1601])
def test_branches_and_slots(branch, depth, n):
    print(f"case voctree sizes <{branch},{depth}> n={n}", flush=True)
    tree, keys = _case(branch, depth, n, branch + n)
    _same(tree, branch, depth, keys)


@pytest.mark.parametrize("tree_exp,key_exp", [(-40, 0), (0, 40), (33, -33), (-59, 59), (-70, 0), (0, 63), (0, -63)])
def test_scales(tree_exp, key_exp):
    print(f"case voctree scales tree 2^{tree_exp} keys 2^{key_exp}", flush=True)
    branch, depth, n = 40, 2, 3000
    tree, keys = _case(branch, depth, n, 5)
    exact = _same(np.ldexp(tree, tree_exp), branch, depth, np.ldexp(keys, key_exp))
    certified = abs(tree_exp) < 60 and abs(key_exp) < 60 and exact < n
    assert certified or exact >= n * depth * 0.5


def test_rows_of_very_different_norm():
    """Keys of every scale in one slot; children whose norms span nine decades."""
    print("case voctree mixed norms", flush=True)
    rng = np.random.default_rng(9)
    branch, depth, n = 50, 2, 4000
    tree, keys = _case(branch, depth, n, 6)
    tree *= (10.0 ** rng.uniform(-9, 0, (tree.shape[0], 1))).astype(np.float32)
    keys *= (2.0 ** rng.integers(-62, 62, (n, 1))).astype(np.float32)
    _same(tree, branch, depth, keys)
