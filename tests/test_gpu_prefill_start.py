"""The first launch of a matrix-core batch (pf_start_kernel: pairs sorted by
expert, tiles listed, rows to operands) at the edges of its range: the largest
batch that takes it (2048 pairs) and the first that does not, the largest of
one workgroup's sort (8192) and the first of the many-workgroup one, the most experts (512), one hot expert that takes half of the pairs
(a tile list of its own, with a remainder), invalid ids (they act as expert
0), and about as many (row, block) units as a workgroup has waves.  Same order and
same bits as the staged kernels."""
import types

import numpy as np
import pytest

from test_gpu_prefill import H, assert_bitexact, batch_run, say  # noqa: F401
from test_gpu_prefill_tiles import random_blocks, rows_with_edges

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tok,topk,n_exp", [(17, 8, 24), (129, 1, 512), (255, 8, 24), (256, 8, 24), (2049, 1, 24), (8192, 1, 3),
                                              (8193, 1, 3)])
def test_start_edges_vs_staged(H, n_tok, topk, n_exp):  # noqa: F811
    rng = np.random.default_rng([n_tok, topk])
    dim = 256
    t = H.Tensor.from_array
    layer = types.SimpleNamespace(gate=t(random_blocks(rng, n_exp * dim, 1, 110)),
                                  up=t(random_blocks(rng, n_exp * dim, 1, 110)),
                                  down=t(random_blocks(rng, n_exp * dim, 1, 84)),
                                  n_expert=n_exp, in_dim=dim, mid_dim=dim, clamp_routed=0.0)
    sel = rng.integers(0, n_exp, (n_tok, topk)).astype(np.int32)
    sel[rng.random((n_tok, topk)) < 0.5] = n_exp - 1
    sel[0, 0], sel[-1, -1] = -1, n_exp
    w = (rng.random((n_tok, topk)) + 0.5).astype(np.float32)
    x = rows_with_edges(rng, n_tok, dim)
    pairs = H.get_option("prefill_min_pairs")
    H.set_option("q8k_min_rows", 0)
    H.set_option("prefill_min_pairs", 128)
    try:
        say(f"start edges {n_tok} x {topk} over {n_exp}: matrix cores")
        a = batch_run(H, layer, sel, w, x, True)
        say(f"start edges {n_tok} x {topk} over {n_exp}: staged")
        b = batch_run(H, layer, sel, w, x, False)
    finally:
        H.set_option("q8k_min_rows", 512)
        H.set_option("prefill_min_pairs", pairs)
    assert a[2] == 2 and b[2] == 0, "matrix-core kernels did not run as selected"
    assert_bitexact(a[1], b[1], "mid mfma vs staged")
    assert_bitexact(a[0], b[0], "out mfma vs staged")
