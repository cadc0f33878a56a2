"""A Q3GU/Q2D shared expert run as one more slot of every token inside the
routed matrix-core launches (batches past the fused decode sizes): the layer
and the FFN block (norm and residual, the combine's residual form) against
the staged kernels bit for bit, with caller selections of K slots, at one
tile, several tiles and a remainder, top-k that has its own combine (8 + 1)
and one that has not."""
import numpy as np
import pytest

from test_gpu_prefill import H, assert_bitexact, map_key  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tok,topk,il", [(33, 8, 10), (64, 8, 44), (130, 3, 43), (301, 8, 10)])
def test_layer_and_block_vs_staged(H, n_tok, topk, il):  # noqa: F811
    from sf37_amd import moe
    D, Fm, E = 1024, 512, 24
    lay = moe.SynthLayer(seed=n_tok, n_expert=E, in_dim=D, mid_dim=Fm, topk=topk, il=il, shared="q3q2")
    w = lay.weights_struct()
    rng = np.random.default_rng(n_tok)
    x = (rng.standard_normal((n_tok, D)) * 3.0).astype(np.float32)
    norm = H.Tensor.from_array(moe.bf16_bits((rng.standard_normal(D) * 0.02).astype(np.float32)))
    key = map_key()
    H.check(H.lib().sf37_hip_register_device_range(key, norm.nbytes, 0, norm.nbytes, norm), "register")
    got = {}
    for mfma in (1, 0):
        H.set_option("prefill_mfma", mfma)
        try:
            xt, out = H.Tensor.from_array(x), H.empty((n_tok, D), np.float32)
            sel, wts = H.empty((n_tok, topk), np.int32), H.empty((n_tok, topk), np.float32)
            print(f"shared slot, {n_tok} tokens, mfma {mfma}: layer", flush=True)
            H.check(H.lib().sf37_hip_moe_layer(out, sel, wts, w, None, xt, n_tok), "layer")
            hid = H.Tensor.from_array(x)
            print(f"shared slot, {n_tok} tokens, mfma {mfma}: block", flush=True)
            H.check(H.lib().sf37_hip_moe_block(hid, None, None, None, w, key, norm.nbytes, 0, 1e-5, None, n_tok), "block")
            got[mfma] = (out.read(np.float32), sel.read(np.int32), wts.read(np.float32), hid.read(np.float32))
        finally:
            H.set_option("prefill_mfma", 1)
    assert (got[1][1] == got[0][1]).all()
    for i, what in ((0, "layer"), (2, "weights"), (3, "block")):
        assert_bitexact(got[1][i], got[0][i], what)
    lay.free()
