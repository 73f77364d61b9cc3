"""float32 products whose operands reach past what the implicit-GEMM kernel addresses with 32-bit offsets: a dense operand of 2 GiB, and a
slice, read in place, whose rows spread over more than that."""
import numpy as np
import pytest

from conftest import closeness

pytestmark = pytest.mark.gpu

# rows, contracted extent, columns: 2.15 GB of lhs, few and very many rows
DENSE = [(131073, 4100, 24), (4300001, 125, 9)]


def build_dense(rows, k, cols):
    """The lhs is made on the device: element (i, k) is (i % 7 + k % 5) / 8, so the product is a sum of two that are small."""
    from jax_mps_amd.shlo.builder import Builder
    b = Builder("gemm_reach")
    w = b.arg((k, cols), "f32")
    lhs = b.add(b.broadcast_in_dim(b.remainder(b.iota((rows,), 0, "i32"), 7), (rows, k), [0]),
                b.broadcast_in_dim(b.remainder(b.iota((k,), 0, "i32"), 5), (rows, k), [1]))
    b.ret(b.matmul(b.mul(b.convert(lhs, "f32"), 0.125), w))
    return b.text()


@pytest.mark.parametrize("rows,k,cols", DENSE)
def test_dense_operand_of_2_gib(client, rows, k, cols):
    from jax_mps_amd import runner
    w = np.random.default_rng(1).uniform(0.1, 1.0, (k, cols)).astype(np.float32)
    print("case dense", rows, k, cols, flush=True)
    got = runner.download(client.compile_and_load(build_dense(rows, k, cols)).execute(runner.upload(client, [w], ["f32"]))[0])
    w = w.astype(np.float64)
    want = 0.125 * ((np.arange(rows) % 7)[:, None] * w.sum(0)[None, :] + ((np.arange(k) % 5) @ w)[None, :])
    # positive terms: a float32 sum of k of them is off by k 2^-24 of itself at the very worst (2.5e-4), by far less in blocks of 16
    ratio = closeness(got, want, 2.5e-4, 1e-6)
    assert ratio <= 1.0, f"{ratio:.3f} x the bound"


WIDE = (8200, 65600)        # 2.15 GB, of which the product reads 512 columns


def build_slice():
    from jax_mps_amd.shlo.builder import Builder
    b = Builder("gemm_reach_slice")
    x, w = b.arg(WIDE, "f32"), b.arg((512, 64), "f32")
    b.ret(b.matmul(b.slice(x, [0, 8], [WIDE[0], 520]), w))
    return b.text()


def test_slice_spread_over_2_gib(client):
    from jax_mps_amd import runner
    rng = np.random.default_rng(2)
    x = np.zeros(WIDE, np.float32)
    x[:, :528] = rng.uniform(-0.1, 0.1, (WIDE[0], 528))
    w = rng.uniform(-0.1, 0.1, (512, 64)).astype(np.float32)
    print("case slice", WIDE, flush=True)
    got = runner.download(client.compile_and_load(build_slice()).execute(runner.upload(client, [x, w], ["f32", "f32"]))[0])
    want = x[:, 8:520].astype(np.float64) @ w.astype(np.float64)
    # 512 products of at most 0.01: float32 sums of them are within 512 2^-24 of 5.12, 1.6e-4, at worst, and in practice within 1e-6
    ratio = closeness(got, want, 1e-5, 1e-5)
    assert ratio <= 1.0, f"{ratio:.3f} x the bound"
