"""The ordered row scatter where its paths can go wrong: single rows and columns, rows of a whole and of no whole number of
four elements, rows larger than a fill workgroup covers, rows named by one update, by a few and by hundreds, update counts
on both sides of the path without a sort (2048) and of the sort in one workgroup (8192), 64-bit indices, a splat operand
(rows without updates are filled, rows with updates start from the splat) and an operand in memory.  Bit for bit against
the updates applied one after the other."""
import numpy as np
import pytest

from shlo_oracle import round_bf16

pytestmark = pytest.mark.gpu

# name, rows, columns, updates, splat operand, dtype, combiner, index dtype
CASES = [
    ("one", 1, 1, 1, True, "f32", "add", "i32"),
    ("no-vector-columns", 7, 3, 15, True, "f32", "add", "i32"),
    ("one-block-of-updates", 5, 6, 64, True, "f32", "add", "i64"),
    ("odd-columns", 600, 37, 255, True, "f32", "add", "i32"),
    ("hot-rows", 600, 36, 2000, True, "f32", "add", "i32"),
    ("several-column-chunks", 513, 1028, 300, True, "f32", "add", "i32"),
    ("several-odd-column-chunks", 40, 259, 300, True, "f32", "max", "i32"),
    ("row-larger-than-a-fill-workgroup", 5, 17000, 40, True, "f32", "add", "i32"),
    ("odd-row-larger-than-a-fill-workgroup", 3, 16387, 20, True, "f32", "add", "i64"),
    ("many-rows", 524288, 4, 1000, True, "f32", "add", "i32"),
    ("last-without-a-sort", 3000, 20, 2048, True, "f32", "add", "i32"),
    ("first-sorted", 3000, 20, 2049, True, "f32", "add", "i32"),
    ("first-radix-sort", 3000, 20, 8193, True, "f32", "add", "i32"),
    ("in-memory", 700, 52, 2048, False, "f32", "add", "i32"),
    ("in-memory-odd", 300, 301, 1500, False, "f32", "max", "i64"),
    ("bf16", 300, 20, 700, True, "bf16", "add", "i32"),
    ("bf16-odd", 300, 21, 700, True, "bf16", "add", "i32"),
]


def build(rows, cols, n, splat, dtype, kind, index):
    from jax_mps_amd.shlo.builder import Builder
    b = Builder("scatter_fold")
    x = b.broadcast_in_dim(b.constant(0.25, dtype), (rows, cols), []) if splat else b.arg((rows, cols), dtype)
    i = b.arg((n,), index)
    u = b.arg((n, cols), dtype)
    b.ret(b.scatter(x, b.reshape(i, (n, 1)), u, update_window_dims=[1], inserted_window_dims=[0],
                    scatter_dims_to_operand_dims=[0], index_vector_dim=1, body=kind))
    return b.text()


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_fold(client, case):
    from jax_mps_amd import runner
    name, rows, cols, n, splat, dtype, kind, index = case
    rng = np.random.default_rng(rows + n)
    idx = (rng.zipf(1.2, size=n) - 1) % (rows + 2)          # a skewed head, the last two values out of range
    idx[::7] = rng.integers(0, rows, size=len(idx[::7]))
    idx = idx.astype(np.int64 if index == "i64" else np.int32)
    idx[5::29] = -1
    operand = np.full((rows, cols), 0.25, np.float32) if splat else rng.standard_normal((rows, cols), dtype=np.float32)
    upd = rng.standard_normal((n, cols), dtype=np.float32)
    if dtype == "bf16":
        operand, upd = round_bf16(operand), round_bf16(upd)
    print("case", name, flush=True)
    ins = [idx, upd] if splat else [operand, idx, upd]
    got = runner.download(client.compile_and_load(build(*case[1:])).execute(
        runner.upload(client, ins, ([index] if splat else [dtype, index]) + [dtype]))[0])
    want = operand.copy()
    ok = (idx >= 0) & (idx < rows)
    if dtype == "bf16":
        for k in np.flatnonzero(ok):
            want[idx[k]] = round_bf16(want[idx[k]] + upd[k])
    else:
        (np.add if kind == "add" else np.maximum).at(want, idx[ok], upd[ok])
    assert np.array_equal(np.asarray(got, np.float32).view(np.uint32), want.view(np.uint32)), name
