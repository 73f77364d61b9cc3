"""Convolutions whose contracted features do not fill whole k-tiles of 16 (the batch of a filter gradient, narrow layers) on the
vector-loader kernel: one short tile, one full and one short tile, features that are and are not multiples of 4 (K-vectors need
the multiple, vectors along the rows do not), split and unsplit K, against the CPU oracle.  The elements past the last feature
of a tap belong to other taps or images: `nan` plants a NaN there, which must reach only the outputs its own products reach."""
import numpy as np
import pytest

from conftest import closeness
from shlo_oracle import Oracle

pytestmark = pytest.mark.gpu

# name, form, batch, height, width, in features, out features, filter, stride, NaN in the first image's corner
CASES = [
    ("wgrad-b24", "wgrad", 24, 9, 10, 48, 32, 3, 1, False),
    ("wgrad-b17", "wgrad", 17, 8, 8, 16, 64, 3, 2, False),
    ("wgrad-b8", "wgrad", 8, 7, 7, 20, 36, 1, 1, False),
    ("wgrad-b31-long", "wgrad", 31, 28, 28, 64, 64, 3, 1, False),
    ("wgrad-b7", "wgrad", 7, 6, 6, 16, 16, 3, 1, False),
    ("fwd-c8", "fwd", 3, 9, 7, 8, 20, 3, 1, False),
    ("fwd-c24", "fwd", 4, 16, 16, 24, 24, 3, 1, False),
    ("fwd-c24-nan", "fwd", 2, 8, 8, 24, 24, 3, 1, True),
    ("fwd-c18", "fwd", 2, 8, 8, 18, 24, 3, 1, False),
    ("dgrad-c40", "dgrad", 2, 9, 9, 24, 40, 3, 1, False),
]


def build(form, b, h, w, cin, cout, k, s, nan):
    from jax_mps_amd.shlo.builder import Builder
    bld = Builder("conv_ragged")
    p = k // 2
    oh, ow = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    if form == "fwd":
        x, f = bld.arg((b, h, w, cin), "f32"), bld.arg((k, k, cin, cout), "f32")
        bld.ret(bld.conv(x, f, strides=(s, s), padding=[[p, p], [p, p]]))
        shapes, K = [x.shape, f.shape], k * k * cin
    elif form == "dgrad":
        g, f = bld.arg((b, oh, ow, cout), "f32"), bld.arg((k, k, cin, cout), "f32")
        bld.ret(bld.conv(g, bld.reverse(f, [0, 1]), strides=(1, 1), padding=[[k - 1 - p] * 2] * 2, dn=("b01f", "01oi", "b01f")))
        shapes, K = [g.shape, f.shape], k * k * cout
    else:
        x, g = bld.arg((b, h, w, cin), "f32"), bld.arg((b, oh, ow, cout), "f32")
        hi = [(o - 1) * s + k - n - p for n, o in ((h, oh), (w, ow))]
        bld.ret(bld.conv(x, g, strides=(1, 1), padding=[[p, hi[0]], [p, hi[1]]], rhs_dilation=(s, s), dn=("f01b", "i01o", "01bf")))
        shapes, K = [x.shape, g.shape], b * oh * ow
    rng = np.random.default_rng(b + h + cin + cout)
    ins = [(rng.uniform(-1, 1, tuple(a)) / np.sqrt(np.sqrt(K))).astype(np.float32) for a in shapes]
    if nan:
        ins[0][0, 0, 1, 0] = np.nan
    return bld.text(), ins


@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_ragged_features(client, case):
    from jax_mps_amd import runner
    name, *spec = case
    text, ins = build(*spec)
    print("case", name, spec, flush=True)
    got = runner.download(client.compile_and_load(text).execute(runner.upload(client, ins, ["f32", "f32"]))[0])
    want = np.asarray(Oracle(text).run(*ins)[0])
    assert np.array_equal(np.isnan(got), np.isnan(want))
    # inputs in [-1, 1] / K^(1/4): results of order 1 / 3 and float32 sums, K 2^-24 of the magnitudes at most
    ratio = closeness(np.nan_to_num(got), np.nan_to_num(want), 1e-5, 1e-5)
    assert ratio <= 1.0, f"{name}: {ratio:.3f} x the bound"
