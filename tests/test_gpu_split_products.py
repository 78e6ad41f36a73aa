"""The fp32 matrix products' split-bf16 form (csrc/gemm_split.hpp: the MLP's backward pair; the tap
and weight-gradient kernels of csrc/conv3x3.hip) at the places where it can go wrong, through the MLP
and conv entry points: K of a partial step only, of whole steps only and of both, output tiles
with one row or column past a tile's edge; operands that the split cannot hold (nonzero under
2^-110), whose tiles are formed again in fp32; and operands that are not finite or round to
infinity in bf16.  Sizes that the rules leave to fp32 MFMAs are among them.  The bar is the fp32
one (1e-5 normwise against the Float32 oracle, with the truth rule), and, where a lost part of
the split must show, one against 64 bits; the split's own error is at most 2^-24 of a product."""
import numpy as np
import pytest

from helpers import ParityCase, make_args, oracle_lib, rel_err, run_parity, to_host

pytestmark = pytest.mark.gpu


def _shapes(size):
    B, I, H, O = size
    sz = dict(loss=1, x=I * B, w1=H * I, b1=H, w2=O * H, b2=O, h1=H * B, z=O * B)
    return {k + suf: v for k, v in sz.items() for suf in ("", "b", "d", "bd")}


def _labels(size):
    return np.arange(size[0], dtype=np.int64) % size[3] + 1


def _scales(size):
    B, I, H, O = size
    g1, g2 = np.sqrt(2.0 / (I + H)), np.sqrt(2.0 / (H + O))
    return {"w1": g1, "w1d": g1, "w2": g2, "w2d": g2, "b1": 0.1, "b2": 0.1}


def _ints(size):
    return dict(zip(("i_b", "i_in", "i_h", "i_out"), size))


@pytest.mark.parametrize("mode", ["b", "d", "hv"])
@pytest.mark.parametrize("size", [(1, 1, 1, 1), (5, 2, 3, 2), (129, 15, 65, 5), (136, 64, 128, 5), (64, 16, 128, 5),
                                  (127, 17, 129, 3), (128, 48, 64, 4), (161, 33, 97, 2)])
def test_split_product_edges(mode, size):
    """Among them operands shorter than a k step's loads, and whole tiles with a partial k step."""
    print(f"mlp2_ce_{mode} {size}", flush=True)
    run_parity("mlp2_ce", mode, _shapes(size), _ints(size), precision="f32", int_arrays=dict(lab=_labels(size)),
               scales=_scales(size))


@pytest.mark.parametrize("mode", ["b", "d", "hv"])
def test_split_product_tiny_operands(mode):
    """x and its direction near 2^-122, below what three bf16 values hold, against weights
    near 2^110: every product is of ordinary size."""
    size = (150, 40, 70, 6)
    s = _scales(size)
    for a in ("x", "xd"):
        s[a] = 2.0 ** -122
    for a in ("w1", "w1d"):
        s[a] *= 2.0 ** 110
    print(f"mlp2_ce_{mode} tiny operands", flush=True)
    run_parity("mlp2_ce", mode, _shapes(size), _ints(size), precision="f32", int_arrays=dict(lab=_labels(size)), scales=s)


@pytest.mark.parametrize("value", [np.inf, np.nan, 3.4e38])
def test_split_product_non_finite(value):
    """One element of x that is not finite, or whose nearest bf16 is infinite (with weights that
    keep its products finite): the same elements of every output are finite as in the oracle,
    the others agree in kind, and the finite ones to the fp32 bar."""
    size = (140, 20, 130, 3)
    s = _scales(size)
    if np.isfinite(value):
        s["w1"] *= 1e-30
    lib = oracle_lib("mlp2_ce", "b", "f32")
    args = make_args(lib, "mlp2_ce_b", _shapes(size), _ints(size), {}, "split-non-finite", np.float32, dict(lab=_labels(size)), s)
    x = next(v for a, _, v in args if a == "x")
    x[7 * size[1] + 3] = value
    host = [v.copy() if isinstance(v, np.ndarray) else v for _, _, v in args]
    lib.call("mlp2_ce_b", *host)
    case = ParityCase("mlp2_ce", "b", args, (), "f32")
    print(f"mlp2_ce_b one element {value}", flush=True)
    case.run_gpu()
    for (a, kind, _), want, dev in zip(args, host, case.dev):
        if kind != "Af":
            continue
        got = to_host(dev)
        assert np.array_equal(np.isnan(got), np.isnan(want)), a
        inf = np.isinf(want)
        assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf]), a
        ok = np.isfinite(want)
        if np.any(want[ok]):
            assert rel_err(got[ok], want[ok]) <= 1e-5, a


def _conv(size):
    N, C, K, H, W = size
    sz = dict(loss=1, xp=(W + 2) * (H + 2) * C * N, w=9 * C * K, out=W * H * K * N)
    return {k + suf: v for k, v in sz.items() for suf in ("", "b", "d", "bd")}, dict(zip(("i_nb", "i_c", "i_k", "i_h", "i_w"), size))


@pytest.mark.parametrize("mode", ["b", "d", "hv"])
@pytest.mark.parametrize("size", [(1, 15, 63, 3, 31), (1, 16, 64, 4, 32), (2, 17, 65, 9, 65), (1, 33, 5, 8, 33), (17, 3, 64, 61, 64)])
def test_split_conv_edges(mode, size):
    """One past and one short of a channel chunk, a row tile, a pixel tile (four-row blocks)."""
    shapes, ints = _conv(size)
    s = 1.0 / np.sqrt(9.0 * size[1])
    print(f"conv3x3_{mode} {size}", flush=True)
    run_parity("conv3x3", mode, shapes, ints, precision="f32", scales={"w": s, "wd": s})


def _tall(cin, r, size):
    """Whether a product with one source takes the eight-row blocks (launch_tap's rule): no fewer
    fp32 steps than six products a tap and chunk, and a block for every CU."""
    import torch
    N, _, _, H, W = size
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return (cin + 1) // 2 >= 6 * ((cin + 15) // 16) and (W + 63) // 64 * N * ((r + 63) // 64) * ((H + 7) // 8) >= cus


@pytest.mark.parametrize("size,scale", [((17, 31, 70, 61, 65), "ordinary"), ((33, 16, 16, 61, 64), "small xp"),
                                        ((33, 16, 16, 61, 64), "small w")])
def test_split_conv_eight_rows(size, scale):
    """The eight-row blocks of the adjoint's forward and of xpb, with a partial last one, ragged
    columns, channels and row tiles; and their fp32 fallback."""
    N, C, K, H, W = size
    assert _tall(C, K, size) and _tall(K, C, size)
    shapes, ints = _conv(size)
    s = 1.0 / np.sqrt(9.0 * C)
    scales = {"w": s, "xp": 1.0}
    if scale != "ordinary":
        small, big = ("xp", "w") if scale == "small xp" else ("w", "xp")
        scales[small] *= 2.0 ** -122
        scales[big] *= 2.0 ** 110
        scales["out"] = scales["outb"] = 2.0 ** -12
    print(f"conv3x3_b {size} {scale}", flush=True)
    run_parity("conv3x3", "b", shapes, ints, precision="f32", scales=scales)


@pytest.mark.parametrize("mode", ["b", "hv"])
@pytest.mark.parametrize("size", [(1, 1, 1, 1, 1), (3, 5, 4, 50, 70), (2, 70, 66, 40, 63), (1, 3, 64, 300, 33), (2, 64, 3, 2, 129)])
def test_split_conv_weight_gradient(mode, size):
    """The weight gradient's strips of 32 and of 64 columns: one pixel, blocks whose rows cross
    strips and images (more rows than blocks), two slabs each way, one past a strip's edge."""
    shapes, ints = _conv(size)
    s = 1.0 / np.sqrt(9.0 * size[1])
    print(f"conv3x3_{mode} {size}", flush=True)
    run_parity("conv3x3", mode, shapes, ints, precision="f32", scales={"w": s, "wd": s})


@pytest.mark.parametrize("mode", ["b", "d", "hv"])
@pytest.mark.parametrize("tiny", ["xp", "w"])
def test_split_conv_tiny_operands(mode, tiny):
    """Images (or weights) near 2^-122 against weights (images) near 2^110."""
    size = (2, 18, 20, 6, 40)
    shapes, ints = _conv(size)
    s = 1.0 / np.sqrt(9.0 * size[1])
    big = {"xp": "w", "w": "xp"}[tiny]
    scales = {"w": s, "wd": s}
    for a, e in ((tiny, -122), (big, 110)):
        for suf in ("", "d"):
            scales[a + suf] = scales.get(a + suf, 1.0) * 2.0 ** e
    # keep every product of ordinary size: out ~ 2^-12, its seeds likewise
    for a in ("out", "outb", "outd", "outbd"):
        scales[a] = 2.0 ** -12
    print(f"conv3x3_{mode} tiny {tiny}", flush=True)
    run_parity("conv3x3", mode, shapes, ints, precision="f32", scales=scales)


@pytest.mark.parametrize("value", [np.inf, 3.4e38])
def test_split_conv_non_finite(value):
    """One pixel that is not finite, or whose nearest bf16 is infinite."""
    size = (1, 5, 9, 7, 40)
    shapes, ints = _conv(size)
    scales = {"w": 1e-20, "outb": 1e-20} if np.isfinite(value) else {}
    lib = oracle_lib("conv3x3", "b", "f32")
    args = make_args(lib, "conv3x3_b", shapes, ints, {}, "split-conv-non-finite", np.float32, None, scales)
    for a, _, v in args:
        if a == "xp":
            v[2 * 9 * 42 + 4 * 42 + 20] = value
        if a == "lossb" and np.isfinite(value):
            v[:] = 1e-37
    host = [v.copy() if isinstance(v, np.ndarray) else v for _, _, v in args]
    lib.call("conv3x3_b", *host)
    case = ParityCase("conv3x3", "b", args, (), "f32")
    print(f"conv3x3_b one pixel {value}", flush=True)
    case.run_gpu()
    for (a, kind, _), want, dev in zip(args, host, case.dev):
        if kind != "Af" or a == "loss":   # (the text's fp32 loss sum overflows where the fp64 one need not)
            continue
        got = to_host(dev)
        assert np.array_equal(np.isnan(got), np.isnan(want)), a
        inf = np.isinf(want)
        assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf]), a
        ok = np.isfinite(want)
        if np.any(want[ok]):
            assert rel_err(got[ok], want[ok]) <= 1e-5, a


@pytest.mark.parametrize("mode,outputs", [("b", ("out", "xpb")), ("d", ("out", "outd")), ("hv", ("out", "outd", "xpb", "xpbd"))])
@pytest.mark.parametrize("size", [(1, 1, 2, 9, 40), (1, 3, 5, 17, 70), (2, 11, 9, 10, 33), (1, 10, 17, 12, 64)])
def test_split_conv_few_channels(mode, outputs, size):
    """Few channels, where the products are summed with fewer roundings: an element is a sum of
    9 c products (the tangents 18 c) rounded at its size at most three times a tap, under
    27 x 2^-24 of the terms' size (1.6e-6), and far less normwise; the seeds that xpb's terms
    hold carry the error of out, its own and that of a product: 3 x 2^-24 more."""
    shapes, ints = _conv(size)
    s = 1.0 / np.sqrt(9.0 * size[1])
    lib = oracle_lib("conv3x3", mode, "f64")
    args = make_args(lib, f"conv3x3_{mode}", shapes, ints, {}, "split-conv-few", np.float32, None, {"w": s, "wd": s})
    host = [v.astype(np.float64) if isinstance(v, np.ndarray) and v.dtype == np.float32 else v for _, _, v in args]
    lib.call(f"conv3x3_{mode}", *host)
    case = ParityCase("conv3x3", mode, args, (), "f32")
    print(f"conv3x3_{mode} {size} few channels", flush=True)
    case.run_gpu()
    for (a, _, _), want, dev in zip(args, host, case.dev):
        if a in outputs:
            assert rel_err(to_host(dev).astype(np.float64), want) <= 1e-6, a


def _bar(n):
    """Largest error over largest value of sums of n products, each rounded at most three times at
    the size of a partial sum by half a unit in its last place (2^-24); such errors add up as the
    root of their number."""
    return np.sqrt(3 * n) * 2.0 ** -24


def _against_64_bits(kernel, mode, shapes, ints, scales, bars, zeros=(), exact=(), int_arrays=None):
    """One generated function, its named outputs against the 64-bit oracle; arrays in `exact`
    hold bf16 values before their scale, and those in `zeros` are zero."""
    lib = oracle_lib(kernel, mode, "f64")
    args = make_args(lib, f"{kernel}_{mode}", shapes, ints, {}, "split-small", np.float32, int_arrays, None)
    for a, kind, v in args:
        if kind != "Af":
            continue
        if a in exact:
            v.view(np.uint32)[...] &= 0xffff0000
        v *= 0.0 if a in zeros else 1.0
        v[...] = (v.astype(np.float64) * scales.get(a, 1.0)).astype(np.float32)
    host = [v.astype(np.float64) if isinstance(v, np.ndarray) and v.dtype == np.float32 else v for _, _, v in args]
    lib.call(f"{kernel}_{mode}", *host)
    case = ParityCase(kernel, mode, args, (), "f32")
    case.run_gpu()
    for (a, _, _), want, dev in zip(args, host, case.dev):
        if a in bars:
            assert np.any(want), a
            e = rel_err(to_host(dev).astype(np.float64), want)
            print(f"{kernel}_{mode} {a} {e:.2e} of {bars[a]:.2e}", flush=True)
            assert e <= bars[a], a


@pytest.mark.parametrize("mode", ["b", "hv"])
def test_split_product_against_64_bits(mode):
    """W1b and xb at K = 784: the split's own error, the rounding of a total a k step and that of D1
    give 1 to 2e-7; without the products l h, h l and m m it would be 4e-6."""
    size = (784, 70, 784, 5)
    s = _scales(size)
    bars = {a: 5e-7 for a in (("w1b", "xb") if mode == "b" else ("w1b", "xb", "w1bd", "xbd"))}
    _against_64_bits("mlp2_ce", mode, _shapes(size), _ints(size), s, bars, ("w1b", "xb", "w1bd", "xbd"), int_arrays=dict(lab=_labels(size)))


# exponents of a whole operand: where the last part of the split is a subnormal (from about 2^-95
# on), both sides of where it no longer holds all bits (2^-110), under fp32's smallest normal (2^-126),
# and wholly under 2^-134, where every part rounds to zero
SMALL = (-98, -106, -109, -111, -122, -130, -141)


@pytest.mark.parametrize("e", SMALL)
@pytest.mark.parametrize("mode", ["b", "hv"])
def test_split_product_small_samples(mode, e):
    """W1b = D1 x' with x near 2^e and D1 near 2^-(20 + e) (the incoming h1b)."""
    size = (150, 40, 70, 6)
    s = {"x": 2.0 ** e, "xd": 2.0 ** e, "h1b": 2.0 ** -(22 + e), "h1bd": 2.0 ** -(22 + e), "w1": 0.1, "w1d": 0.1, "w2": 0.2, "w2d": 0.2}
    bars = {a: _bar(size[0]) for a in (("w1b",) if mode == "b" else ("w1b", "w1bd"))}
    _against_64_bits("mlp2_ce", mode, _shapes(size), _ints(size), s, bars, ("w1b", "w1bd"), int_arrays=dict(lab=_labels(size)))


@pytest.mark.parametrize("e", SMALL)
@pytest.mark.parametrize("mode", ["b", "hv"])
def test_split_product_small_weights(mode, e):
    """xb = W1' D1 with W1 near 2^e and D1 near 2^-(20 + e)."""
    size = (150, 40, 70, 6)
    s = {"w1": 2.0 ** e, "w1d": 2.0 ** e, "h1b": 2.0 ** -(22 + e), "h1bd": 2.0 ** -(22 + e), "w2": 0.2, "w2d": 0.2}
    bars = {a: _bar(size[2]) for a in (("xb",) if mode == "b" else ("xb", "xbd"))}
    _against_64_bits("mlp2_ce", mode, _shapes(size), _ints(size), s, bars, ("xb", "xbd"), int_arrays=dict(lab=_labels(size)))


@pytest.mark.parametrize("e,exact", [(e, False) for e in SMALL] + [(-115, True), (-131, True)])
@pytest.mark.parametrize("size", [(2, 10, 17, 6, 40), (2, 18, 20, 6, 40)])
@pytest.mark.parametrize("product", ["out by xp", "out by w", "xpb by g", "xpb by w", "wb by xp", "wb by g"])
def test_split_conv_small(product, size, e, exact):
    """Each product of the adjoint with one operand near 2^e and the other near 2^-(20 + e); exact:
    bf16 values, which the split holds down to its subnormals.  (lossb = 0 where g is small or
    large on its own: g is then outb.)"""
    N, C, K, H, W = size
    shapes, ints = _conv(size)
    out, _, by = product.split()
    other = {"out": {"xp": "w", "w": "xp"}, "xpb": {"g": "w", "w": "g"}, "wb": {"xp": "g", "g": "xp"}}[out][by]
    name = lambda a: "outb" if a == "g" else a  # noqa: E731
    scales = {name(by): 2.0 ** e, name(other): 2.0 ** -(22 + e)}
    zeros = ("out", "xpb", "wb") + (("lossb",) if out != "out" else ())
    n = {"out": 9 * C, "xpb": 9 * K, "wb": N * H * W}[out]
    _against_64_bits("conv3x3", "b", shapes, ints, scales, {out: _bar(n)}, zeros, (name(by),) if exact else ())


@pytest.mark.parametrize("e", SMALL)
@pytest.mark.parametrize("size", [(2, 10, 17, 6, 40), (2, 18, 20, 6, 40)])
@pytest.mark.parametrize("by", ["g", "w"])
def test_split_conv_small_two_sources(by, size, e):
    """xpb and xpbd of the HVP (two products to an element of xpbd), as above."""
    shapes, ints = _conv(size)
    scales = {a + s: 2.0 ** (e if a[0] == ("o" if by == "g" else "w") else -(22 + e)) for a, s in (("outb", ""), ("outb", "d"), ("w", ""), ("w", "d"))}
    bars = {a: _bar(18 * size[2]) for a in ("xpb", "xpbd")}
    _against_64_bits("conv3x3", "hv", shapes, ints, scales, bars, ("xpb", "xpbd", "lossb", "lossbd"))


@pytest.mark.parametrize("row", [3, 70, 129])
@pytest.mark.parametrize("product", ["out", "xpb", "xpbd"])
def test_split_conv_small_row(product, row):
    """One output row (of three row tiles) whose weights are near 2^-120, against pixels near 2^98;
    for xpbd only the direction's: a block must notice its own row tile's, of either set."""
    N, C, K, H, W = size = (1, 6, 131, 5, 33) if product == "out" else (1, 131, 6, 5, 33)
    shapes, ints = _conv(size)
    mode = "hv" if product == "xpbd" else "b"
    lib = oracle_lib("conv3x3", mode, "f64")
    args = make_args(lib, f"conv3x3_{mode}", shapes, ints, {}, "split-row", np.float32, None,
                     {a: 2.0 ** 98 for a in ("xp", "outb", "outbd")} if product != "out" else {"xp": 2.0 ** 98})
    v = {a: x for a, _, x in args}
    for a in ("xpb", "xpbd", "out", "lossb", "lossbd") if product != "out" else ("out",):
        if a in v:
            v[a][...] = 0.0
    if product != "out":
        v["xp"] *= np.float32(2.0 ** -98)
    pick = (lambda a: a.reshape(K, C, 9)[row]) if product == "out" else (lambda a: a.reshape(K, C, 9)[:, row])
    for a in ("w", "wd"):
        if a in v:
            pick(v[a])[...] *= np.float32(0.0 if (product == "xpbd" and a == "w") else 2.0 ** -120)
    host = [x.astype(np.float64) if isinstance(x, np.ndarray) and x.dtype == np.float32 else x for _, _, x in args]
    lib.call(f"conv3x3_{mode}", *host)
    case = ParityCase("conv3x3", mode, args, (), "f32")
    print(f"conv3x3_{mode} {product} row {row}", flush=True)
    case.run_gpu()
    for (a, _, _), want, dev in zip(args, host, case.dev):
        if a == product:
            rows = lambda x: x.reshape((N, K, H, W) if product == "out" else (N, C, H + 2, W + 2))[:, row]  # noqa: E731
            want, got = rows(want), rows(to_host(dev).astype(np.float64))
            if product != "out":   # (the frame is border_kernel's)
                want, got = want[:, 1:-1, 1:-1], got[:, 1:-1, 1:-1]
            assert np.any(want) and rel_err(got, want) <= _bar(9 * (C if product == "out" else K)), a
