"""The bf16 product kernel for few output tiles (a workgroup per 16 to 64 rows and 32 columns, K shared out to its wavefronts):
one row, ragged rows and columns, each number of row blocks, K of one slab, of fewer slabs than wavefronts, of a slab count
that does not divide and of many slabs, both layouts of the right-hand side, bias, float32 results, a batch dim, and the
largest grids it takes next to the first it leaves to the ring kernel (64 rows a workgroup from K = 768 on)."""
import numpy as np
import pytest

from conftest import closeness
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
