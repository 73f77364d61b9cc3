"""The bf16 product kernel for few output tiles (a workgroup per 16 to 64 rows and 32 columns, K shared out to its wavefronts):
one row, ragged rows and columns, each number of row blocks, K of one slab, of fewer slabs than wavefronts, of a slab count
that does not divide and of many slabs, both layouts of the right-hand side, bias, float32 results, a batch dim, and the
largest grids it takes next to the first it leaves to the ring kernel (64 rows a workgroup from K = 768 on)."""
import os

import numpy as np
import pytest

import op_cases
from conftest import closeness
from test_gpu_ops import test_op_case as check_op_case
from shlo_oracle import Oracle, round_bf16
from test_gpu_gemm_wide import build

pytestmark = pytest.mark.gpu

NN, NT = ([1], [0]), ([1], [1])
# name, lhs shape, rhs shape, contracting dims (lhs, rhs), batch dims, bias, out dtype
CASES = [
    ("one-row", (1, 32), (32, 8), NN, ((), ()), True, "bf16"),
    ("rows-17-k-96", (17, 96), (96, 40), NN, ((), ()), True, "bf16"),
    ("rows-37-k-416", (37, 416), (416, 776), NN, ((), ()), True, "bf16"),
    ("rows-37-long-k", (37, 3072), (3072, 768), NN, ((), ()), True, "bf16"),
    ("two-blocks", (95, 160), (160, 2056), NN, ((), ()), False, "bf16"),
    ("three-blocks", (96, 64), (64, 4096), NN, ((), ()), True, "bf16"),
    ("four-blocks-largest", (64, 96), (96, 8192), NN, ((), ()), False, "bf16"),
    # four and more slabs of K per wavefront, with remainders, for each number of row blocks and both layouts
    ("two-blocks-long-k", (37, 800), (800, 3072), NN, ((), ()), True, "bf16"),
    ("three-blocks-long-k", (96, 864), (864, 4096), NN, ((), ()), True, "bf16"),
    ("four-blocks-long-k", (64, 928), (928, 8192), NN, ((), ()), True, "bf16"),
    ("two-blocks-long-k-nt", (37, 832), (3072, 832), NT, ((), ()), True, "bf16"),
    ("three-blocks-long-k-nt", (96, 896), (4090, 896), NT, ((), ()), False, "bf16"),
    ("four-blocks-long-k-nt", (63, 800), (8192, 800), NT, ((), ()), True, "f32"),
    ("four-blocks-short-k", (64, 736), (736, 8192), NN, ((), ()), True, "bf16"),
    ("three-blocks-nt-short-k", (96, 512), (4096, 512), NT, ((), ()), False, "bf16"),
    ("three-blocks-nt", (96, 768), (4096, 768), NT, ((), ()), False, "bf16"),
    ("past-the-line", (65, 128), (128, 8192), NN, ((), ()), False, "bf16"),
    ("nt-odd-columns", (33, 224), (33, 224), NT, ((), ()), False, "bf16"),
    ("nt-f32-odd-columns", (50, 192), (45, 192), NT, ((), ()), True, "f32"),
    ("nn-f32", (50, 1056), (1056, 72), NN, ((), ()), False, "f32"),
    ("batched", (3, 20, 96), (3, 96, 72), ([2], [1]), ([0], [0]), False, "bf16"),
]


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_few_tiles(client, case):
    from jax_mps_amd import runner
    name, *spec = case
    text, shapes, dtypes = build(*spec)
    rng = np.random.default_rng(len(name))
    ins = [rng.standard_normal(s).astype(np.float32) for s in shapes]
    print("case", name, spec, flush=True)
    got = runner.download(client.compile_and_load(text).execute(runner.upload(client, ins, dtypes))[0])
    want = Oracle(text).run(*[round_bf16(a) if d == "bf16" else a for a, d in zip(ins, dtypes)])[0]
    # bf16: two roundings (product, sum with the bias) of 2^-9 each and float32 sums; float32: K products in float32,
    # K 2^-24 of the sum of their magnitudes at most, which is below 1e-5 of the largest result at these K
    f32 = spec[-1] == "f32"
    ratio = closeness(got, want, 1e-5 if f32 else 2e-2, 1e-5 * float(np.abs(want).max()) if f32 else 2e-2)
    assert ratio <= 1.0, f"{name}: {ratio:.3f} x the bound"


# the kernels that this one takes most small products from (the 64x64 tiles of the ring kernel, and the tiled kernel behind it):
# edges, layouts, batches and epilogues
BEHIND = [n for n in op_cases.case_names() if n.startswith(("dot-bf16-", "dot-bias-bf16-", "dot-gelu-bf16-"))]


@pytest.mark.parametrize("name", BEHIND)
def test_the_kernels_behind_it(client, name):
    os.environ["MI355X_GEMM_FEW"] = "0"
    try:
        check_op_case(client, name)
    finally:
        del os.environ["MI355X_GEMM_FEW"]


# a GELU in the epilogue, one to four row blocks a workgroup
GELU = [("one-block", 37, 800, 768), ("two-blocks", 37, 800, 3072), ("three-blocks", 96, 800, 4096), ("four-blocks", 64, 800, 8192)]


def build_gelu(rows, k, cols):
    from jax_mps_amd.shlo.builder import Builder, gelu_tanh
    b = Builder("gemm_few_gelu")
    x, w, v = b.arg((rows, k), "bf16"), b.arg((k, cols), "bf16"), b.arg((cols,), "bf16")
    y = b.matmul(x, w)
    b.ret(gelu_tanh(b, b.add(y, b.broadcast_in_dim(v, y.shape, [1]))))
    return b.text(), [(rows, k), (k, cols), (cols,)]


@pytest.mark.parametrize("case", GELU, ids=[c[0] for c in GELU])
def test_gelu(client, case):
    from jax_mps_amd import runner
    name, *spec = case
    text, shapes = build_gelu(*spec)
    rng = np.random.default_rng(len(name))
    ins = [(rng.standard_normal(s) * 0.3).astype(np.float32) for s in shapes]
    print("case", name, spec, flush=True)
    got = runner.download(client.compile_and_load(text).execute(runner.upload(client, ins, ["bf16"] * 3))[0])
    want = Oracle(text).run(*[round_bf16(a) for a in ins])[0]
    # as for the products above: the epilogue rounds the product, the sum and the activation, 2^-9 each
    ratio = closeness(got, want, 2e-2, 2e-2)
    assert ratio <= 1.0, f"{name}: {ratio:.3f} x the bound"
