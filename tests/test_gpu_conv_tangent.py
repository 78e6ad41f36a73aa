"""conv3x3's tangent forward (tangent and HVP: out, outd, loss, lossd) against its fp32 chain: per
element, channels in pairs (two fused multiply-adds), the nine taps of a pair in order; outd
adds wd xp before w xpd.  lossd sums products of out and outd that cancel, so its relative error is
theirs times a condition number of 10 to 100 and more: another order of rounding moves it past
5e-6 for some inputs.  out and outd are therefore held to the chain bit for bit, and loss
and lossd to the fp64 sum of its terms, rounded once (2^-24) and summed in another order
(1e-13 of the terms' magnitudes)."""
import numpy as np
import pytest

from helpers import ParityCase, make_args, oracle_lib, to_host

pytestmark = pytest.mark.gpu


def _fma(acc, a, b):
    # a product of two float32 is exact in float64, and its sum with a third nearly so in 80 bits
    return (acc.astype(np.longdouble) + a.astype(np.float64) * b.astype(np.float64)).astype(np.float32)


def _chain(xp, w, xpd, wd, H, W):
    N, C, K = xp.shape[0], xp.shape[1], w.shape[0]
    out, outd = np.zeros((N, K, H, W), np.float32), np.zeros((N, K, H, W), np.float32)
    pixels = lambda a, c, ky, kx: a[:, None, c, ky:ky + H, kx:kx + W]  # noqa: E731
    weights = lambda a, c, ky, kx: a[None, :, c, ky, kx, None, None]  # noqa: E731
    for c in range(0, C, 2):
        pair = range(c, min(c + 2, C))
        for ky in range(3):
            for kx in range(3):
                for q in pair:
                    out = _fma(out, weights(w, q, ky, kx), pixels(xp, q, ky, kx))
                for q in pair:
                    outd = _fma(outd, weights(wd, q, ky, kx), pixels(xp, q, ky, kx))
                for q in pair:
                    outd = _fma(outd, weights(w, q, ky, kx), pixels(xpd, q, ky, kx))
    return out, outd


@pytest.mark.parametrize("mode", ["d", "hv"])
@pytest.mark.parametrize("size", [(1, 1, 1, 1, 1), (2, 3, 5, 7, 70), (2, 18, 66, 6, 40), (1, 32, 48, 22, 50), (4, 33, 7, 9, 65)])
def test_conv_tangent_is_the_fp32_chain(mode, size):
    N, C, K, H, W = size
    sz = dict(loss=1, xp=(W + 2) * (H + 2) * C * N, w=9 * C * K, out=W * H * K * N)
    shapes = {k + suf: v for k, v in sz.items() for suf in ("", "b", "d", "bd")}
    ints = dict(zip(("i_nb", "i_c", "i_k", "i_h", "i_w"), size))
    s = 1.0 / np.sqrt(9.0 * C)
    lib = oracle_lib("conv3x3", mode, "f32")
    args = make_args(lib, f"conv3x3_{mode}", shapes, ints, {}, "conv-tangent", np.float32, None, {"w": s, "wd": s})
    v = {a: x for a, _, x in args}
    xs, ws = (N, C, H + 2, W + 2), (K, C, 3, 3)
    out, outd = _chain(v["xp"].reshape(xs), v["w"].reshape(ws), v["xpd"].reshape(xs), v["wd"].reshape(ws), H, W)
    print(f"conv3x3_{mode} {size} tangent forward", flush=True)
    case = ParityCase("conv3x3", mode, args, (), "f32")
    case.run_gpu()
    got = {a: to_host(d) for (a, kind, _), d in zip(args, case.dev) if kind == "Af"}
    assert np.array_equal(got["out"], out.ravel())
    assert np.array_equal(got["outd"], outd.ravel())
    o, od = out.ravel().astype(np.float64), outd.ravel().astype(np.float64)
    for a, terms in (("loss", 0.5 * o * o), ("lossd", o * od)):
        want = float(v[a][0]) + terms.sum()
        assert abs(float(got[a][0]) - want) <= 2.0 ** -24 * abs(want) + 1e-13 * np.abs(terms).sum(), a
