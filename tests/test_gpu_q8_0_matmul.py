"""Q8_0 products of many tokens on the int8 matrix cores (k_prefill.hip
sh_gemm) against the dot-product kernel, bit for bit, through
matmul_q8_0_mapped and matmul_q8_0_pair_mapped: column tiles that are whole,
partial or a single column (64 and 128 columns per workgroup), token tiles
of 64 with remainders, one and two matrices, the batch sizes around the rule
that chooses between the two kernels."""
import numpy as np
import pytest

from test_gpu_prefill import H, assert_bitexact, map_key  # noqa: F401

pytestmark = pytest.mark.gpu


def products(H, K, N, T, pair, x, w, mfma):  # noqa: F811
    L = H.lib()
    key, nb = map_key(), w[0].nbytes
    for i, t in enumerate(w):
        H.check(L.sf37_hip_register_device_range(key, 2 * nb, i * nb, nb, t), "register")
    out = [H.Tensor.from_array(np.full((T, N), np.nan, np.float32)) for _ in range(2)]
    xt = H.Tensor.from_array(x)
    H.set_option("prefill_mfma", mfma)
    L.sf37_hip_profile_enable(1)
    H.profile_read()
    try:
        if pair:
            H.check(L.sf37_hip_matmul_q8_0_pair_mapped(out[0], out[1], key, 2 * nb, 0, nb, K, N, xt, T), "pair")
        else:
            H.check(L.sf37_hip_matmul_q8_0_mapped(out[0], key, 2 * nb, 0, K, N, xt, T), "matmul")
        H.profile_read()
    finally:
        L.sf37_hip_profile_enable(0)
        H.set_option("prefill_mfma", 1)
    return [o.read(np.float32) for o in out[:2 if pair else 1]]


@pytest.mark.parametrize("K,N,T,pair", [
    (4096, 1280, 19, True), (4096, 1280, 20, True), (1280, 4096, 20, False), (4096, 288, 85, False),
    (4096, 288, 86, False), (256, 129, 191, False), (512, 1, 24577, False), (256, 100, 300, True),
    (1280, 4096, 1100, False), (256, 130, 5000, True)])
def test_matmul_q8_0_matrix_cores(H, K, N, T, pair):  # noqa: F811
    w = [H.synth_quant("q8_0", N, K, 5, s) for s in (1, 2)]
    rng = np.random.default_rng([K, N, T])
    x = rng.standard_normal((T, K)).astype(np.float32)
    x[:, :32] = 0.0
    x[::3, 32:64] *= 1e4
    print(f"q8_0 products {K} -> {N}, {T} tokens", flush=True)
    a, b = products(H, K, N, T, pair, x, w, 1), products(H, K, N, T, pair, x, w, 0)
    for i, (g, h) in enumerate(zip(a, b)):
        assert np.isfinite(g).all(), "an output was not written"
        assert_bitexact(g, h, f"matrix {i}")
