"""mlp2_ce's forward products (h1; tangent and HVP: h1d too) against their fp32 chain: k in groups
of eight, pairs (k, k + 4) of a group in order, one fused multiply-add each; the tangent's
W1 xd before W1d x.  W1 is scaled so that s1 is near 1e-6, where tanh(s1) = s1 and
1 - h1^2 = 1 in fp32, and the biases are zero: h1 and h1d are then the products themselves and are
held bit for bit.  (lossd sums terms that cancel, and the bias gradients sum over the batch: another
order of rounding in the forward shows there many times enlarged.)"""
import numpy as np
import pytest

from helpers import ParityCase, make_args, oracle_lib, to_host

pytestmark = pytest.mark.gpu


def _fma(acc, a, b):
    # a product of two float32 is exact in float64, and its sum with a third nearly so in 80 bits
    return (acc.astype(np.longdouble) + a.astype(np.float64) * b.astype(np.float64)).astype(np.float32)


@pytest.mark.parametrize("mode", ["b", "d", "hv"])
@pytest.mark.parametrize("size", [(1, 1, 1, 1), (130, 40, 70, 3), (64, 200, 129, 5), (33, 17, 128, 2), (128, 64, 64, 4)])
def test_mlp_forward_is_the_fp32_chain(mode, size):
    B, I, H, O = size
    sz = dict(loss=1, x=I * B, w1=H * I, b1=H, w2=O * H, b2=O, h1=H * B, z=O * B)
    shapes = {k + suf: v for k, v in sz.items() for suf in ("", "b", "d", "bd")}
    lib = oracle_lib("mlp2_ce", mode, "f32")
    args = make_args(lib, f"mlp2_ce_{mode}", shapes, dict(zip(("i_b", "i_in", "i_h", "i_out"), size)), {}, "mlp-forward", np.float32,
                     dict(lab=np.arange(B, dtype=np.int64) % O + 1), {"w1": 2.0 ** -20 / np.sqrt(I), "b1": 0.0, "b1d": 0.0})
    v = {a: x for a, _, x in args}
    x, w = v["x"].reshape(B, I), v["w1"].reshape(I, H)     # column-major (I, B) and (H, I)
    s = np.zeros((B, H), np.float32)
    sd = np.zeros((B, H), np.float32)
    # a group's pair (k, k + 4) is one instruction: both of W1 xd, then both of W1d x
    groups = [[k for k in (g + c, g + c + 4) if k < I] for g in range(0, I, 8) for c in range(4)]
    for ks in groups:
        for k in ks:
            s = _fma(s, x[:, k:k + 1], w[k:k + 1])
        if mode != "b":
            xd, wd = v["xd"].reshape(B, I), v["w1d"].reshape(I, H)
            for k in ks:
                sd = _fma(sd, xd[:, k:k + 1], w[k:k + 1])
            for k in ks:
                sd = _fma(sd, x[:, k:k + 1], wd[k:k + 1])
    print(f"mlp2_ce_{mode} {size} forward", flush=True)
    case = ParityCase("mlp2_ce", mode, args, (), "f32")
    case.run_gpu()
    got = {a: to_host(d) for (a, kind, _), d in zip(args, case.dev) if kind == "Af"}
    assert np.array_equal(got["h1"], s.ravel())
    if mode != "b":
        assert np.array_equal(got["h1d"], sd.ravel())
