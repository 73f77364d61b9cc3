"""float32 products whose operands reach past what the implicit-GEMM kernel addresses with 32-bit offsets: a dense operand of 2 GiB."""
import numpy as np
import pytest

from conftest import closeness

pytestmark = pytest.mark.gpu

ROWS, K, N = 131073, 4100, 24       # 2.15 GB of lhs


def build_dense():
    """The lhs is made on the device: element (i, k) is (i % 7 + k % 5) / 8, so the product is a sum of two that are small."""
    from jax_mps_amd.shlo.builder import Builder
    b = Builder("gemm_reach")
    w = b.arg((K, N), "f32")
    lhs = b.add(b.broadcast_in_dim(b.remainder(b.iota((ROWS,), 0, "i32"), 7), (ROWS, K), [0]),
                b.broadcast_in_dim(b.remainder(b.iota((K,), 0, "i32"), 5), (ROWS, K), [1]))
    b.ret(b.matmul(b.mul(b.convert(lhs, "f32"), 0.125), w))
    return b.text()


def test_dense_operand_of_2_gib(client):
    from jax_mps_amd import runner
    w = np.random.default_rng(1).uniform(0.1, 1.0, (K, N)).astype(np.float32)
    print("case dense", ROWS, K, N, flush=True)
    got = runner.download(client.compile_and_load(build_dense()).execute(runner.upload(client, [w], ["f32"]))[0])
    w = w.astype(np.float64)
    want = 0.125 * ((np.arange(ROWS) % 7)[:, None] * w.sum(0)[None, :] + ((np.arange(K) % 5) @ w)[None, :])
    # positive terms: a float32 sum of K of them is off by K 2^-24 of itself at the very worst (2.5e-4), by far less in blocks of 16
    ratio = closeness(got, want, 2.5e-4, 1e-6)
    assert ratio <= 1.0, f"{ratio:.3f} x the bound"
