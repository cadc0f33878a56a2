"""The matrix-core routed kernels at the edges of their tiles (k_prefill.hip).

Groups of 1, 31, 32, 33, 63, 64, 65 and 129 pairs (a tile holds up to 64, as
one or two 32-pair blocks; one more expert is idle), rows of one to five
256-blocks (the block loop's ends, and Q3 blocks that start on and between
dwords), weights of random bytes (every code and zero point, header bits the
format ignores, scales of both signs) and rows whose blocks quantise to every
code from -128 (saturated: a subnormal block) to 127, or to zero.  The group
sums are exact integers and the float epilogue has one order, so the outputs
equal the staged dot-product kernels' bit for bit.
"""
import types

import numpy as np
import pytest

from test_gpu_prefill import H, assert_bitexact, batch_run, say  # noqa: F401

pytestmark = pytest.mark.gpu

GROUPS = [1, 31, 32, 33, 0, 63, 64, 65, 129]


def random_blocks(rng, rows, nblk, size):
    b = rng.integers(0, 256, (rows, nblk, size), dtype=np.uint8)
    s = (rng.standard_normal((rows, nblk, 4)) * 0.01).astype(np.float16)
    b[..., :8] = s.view(np.uint8).reshape(rows, nblk, 8)
    return b.reshape(-1)


def rows_with_edges(rng, n, dim):
    x = rng.standard_normal((n, dim // 256, 256)).astype(np.float32)
    x[0::7, 0] = 0.0                                       # an all-zero block
    x[1::7, 0] *= np.float32(1e-39)                        # 1 / d overflows: codes saturate at -128 and 127
    x[2::7, -1, :] = np.where(rng.random((len(x[2::7]), 256)) < 0.5, 3.0, -3.0)   # all codes at +-127
    x[3::7, -1, :64] = 100.0                               # a group of 127s beside small codes
    return x.reshape(n, dim)


@pytest.mark.parametrize("in_dim,mid_dim", [(256, 256), (512, 1280), (768, 512), (1024, 768), (1280, 1024)])
def test_tile_edges_vs_staged(H, in_dim, mid_dim):  # noqa: F811
    rng = np.random.default_rng([in_dim, mid_dim])
    n_exp, n_tok = len(GROUPS), sum(GROUPS)
    t = H.Tensor.from_array
    layer = types.SimpleNamespace(
        gate=t(random_blocks(rng, n_exp * mid_dim, in_dim // 256, 110)),
        up=t(random_blocks(rng, n_exp * mid_dim, in_dim // 256, 110)),
        down=t(random_blocks(rng, n_exp * in_dim, mid_dim // 256, 84)),
        n_expert=n_exp, in_dim=in_dim, mid_dim=mid_dim, clamp_routed=0.0)
    sel = rng.permutation(np.repeat(np.arange(n_exp), GROUPS)).astype(np.int32)[:, None]
    w = (rng.random((n_tok, 1)) + 0.5).astype(np.float32)
    x = rows_with_edges(rng, n_tok, in_dim)
    H.set_option("q8k_min_rows", 0)
    try:
        say(f"tile edges in {in_dim} mid {mid_dim}: matrix cores")
        a = batch_run(H, layer, sel, w, x, True)
        say(f"tile edges in {in_dim} mid {mid_dim}: staged")
        b = batch_run(H, layer, sel, w, x, False)
    finally:
        H.set_option("q8k_min_rows", 512)
    assert a[2] == 2 and b[2] == 0, "matrix-core kernels did not run as selected"
    assert_bitexact(a[1], b[1], "mid mfma vs staged")
    assert_bitexact(a[0], b[0], "out mfma vs staged")
    assert np.isfinite(a[0]).all() and np.abs(a[0]).max() > 0
