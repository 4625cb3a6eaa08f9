"""The N-D executor (NdGraph, src/nd.rs) on the GPU against the oracle, through the C ABI
(ocr_nd_*): every fusion pattern and operator on small graphs, then the PP-OCRv6-architecture
recogniser (36 lines, widths in [160, 960]) and the DB detector's front end and map.

Tolerances: float32 activations go through the matrix cores as float16 hi + lo (about 2^-22
relative), so results agree with the float32 oracle to float32 rounding:
|gpu - oracle| <= 1e-4 * (1 + |oracle|) per operator. Recognition: the identical arg-max at every
CTC step and probabilities within 1e-3. Detection: probabilities within 1e-4, so the thresholded
mask is bit-exact outside the 1e-4 band around the threshold."""
import numpy as np
import pytest

from ocrhip import onnx_write as ow
from ocrhip import synth_pp
from oracle import graph as og
from oracle import onnx_read

pytestmark = pytest.mark.gpu
RNG = np.random.Generator(np.random.PCG64(91))


def f16x(a):
    return np.asarray(a, np.float32).astype(np.float16).astype(np.float32)


def build(tmp_path, name, fn, in_shape):
    g = ow.Graph(name)
    out = fn(g, "x")
    p = tmp_path / f"{name}.onnx"
    p.write_bytes(g.model("x", list(in_shape), out, ["a"] * 1))
    return str(p)


def check(ctx, path, x, tol=1e-4, stop=False):
    import ocrhip
    print(f"nd graph {path} input {x.shape}", flush=True)
    got = ocrhip.NdGraph(ctx, path, stop).run(x)
    want, _ = og.run(onnx_read.load(path), x)
    assert got.shape == want.shape, (got.shape, want.shape)
    err = np.abs(got - want) / (1 + np.abs(want))
    assert err.max() <= tol, f"max rel err {err.max()}"
    return got, want


def ran(names, fn):
    """Runs fn with the kernel families or forms probed; returns {name: launches}."""
    import ocrhip
    for f in names:
        ocrhip.probe_start(f)
    fn()
    return {f: ocrhip.probe_stop(f)["calls"] for f in names}


def w(g, shape, fan, exact=True):
    a = RNG.standard_normal(shape).astype(np.float32) * np.float32(np.sqrt(2 / fan))
    return g.init(g.fresh("w"), f16x(a) if exact else a)


def conv(g, x, cin, cout, k=3, stride=(1, 1), group=1, bias=True, exact=True):
    ins = [x, w(g, (cout, cin // group, k, k), cin // group * k * k, exact)]
    if bias:
        ins.append(g.init(g.fresh("b"), (RNG.standard_normal(cout) * 0.1).astype(np.float32)))
    return g.add("Conv", ins, kernel_shape=[k, k], pads=[k // 2] * 4, strides=list(stride), group=group)


def bn(g, x, c):
    vals = [RNG.uniform(0.8, 1.2, c), RNG.uniform(-.1, .1, c), RNG.uniform(-.1, .1, c), RNG.uniform(.5, 1.5, c)]
    return g.add("BatchNormalization", [x] + [g.init(g.fresh("bn"), v.astype(np.float32)) for v in vals], epsilon=1e-5)


def const(g, v):
    return g.init(g.fresh("c"), np.array([v], np.float32))


def ints(g, v):
    return g.init(g.fresh("i"), np.array(v, np.int64))


def test_conv_bn_relu_nchw_mfma(ctx, tmp_path):
    p = build(tmp_path, "cbr", lambda g, x: g.add("Relu", [bn(g, conv(g, x, 24, 40, bias=False), 40)]), (2, 24, 11, 29))
    check(ctx, p, RNG.standard_normal((2, 24, 11, 29)).astype(np.float32))


def test_conv_bias_add_and_1x1(ctx, tmp_path):
    def fn(g, x):
        y = conv(g, x, 16, 32, k=1, bias=False)
        y = g.add("Add", [y, g.init("ab", (RNG.standard_normal((1, 32, 1, 1)) * 0.1).astype(np.float32))])
        return g.add("Relu", [y])
    p = build(tmp_path, "cba", fn, (1, 16, 6, 45))
    check(ctx, p, RNG.standard_normal((1, 16, 6, 45)).astype(np.float32))


def test_strided_and_depthwise_convs(ctx, tmp_path):
    def fn(g, x):
        y = g.add("Relu", [bn(g, conv(g, x, 3, 16, stride=(2, 2), bias=False), 16)])
        y = g.add("Relu", [conv(g, y, 16, 16, group=16)])
        return g.add("Relu", [bn(g, conv(g, y, 16, 16, stride=(2, 1), group=16, bias=False), 16)])
    p = build(tmp_path, "sd", fn, (2, 3, 24, 40))
    check(ctx, p, RNG.standard_normal((2, 3, 24, 40)).astype(np.float32))


def test_se_gate_gelu_residual(ctx, tmp_path):
    def fn(g, x):
        se = g.add("GlobalAveragePool", [x])
        se = g.add("Relu", [conv(g, se, 32, 8, k=1)])
        se = g.add("HardSigmoid", [conv(g, se, 8, 32, k=1)], alpha=0.2, beta=0.5)
        y = g.add("Mul", [x, se])
        y = conv(g, y, 32, 32, k=1)
        d = g.add("Div", [y, const(g, np.float32(np.sqrt(2.0)))])
        e = g.add("Erf", [d])
        a = g.add("Add", [e, const(g, 1.0)])
        m = g.add("Mul", [y, a])
        y = g.add("Mul", [m, const(g, 0.5)])
        return g.add("Add", [y, x])
    p = build(tmp_path, "seg", fn, (2, 32, 3, 17))
    check(ctx, p, RNG.standard_normal((2, 32, 3, 17)).astype(np.float32))


def test_hardsigmoid_non_default_attributes(ctx, tmp_path):
    # The SE gate with torch's hardsigmoid constants (alpha 1/6) and a standalone HardSigmoid with
    # alpha 0.3, beta 0.4: the attributes, not ONNX's defaults, reach the kernels.
    def fn(g, x):
        se = g.add("GlobalAveragePool", [x])
        se = g.add("HardSigmoid", [conv(g, se, 32, 32, k=1)], alpha=1.0 / 6.0, beta=0.5)
        y = conv(g, g.add("Mul", [x, se]), 32, 32, k=1)
        return g.add("HardSigmoid", [y], alpha=0.3, beta=0.4)
    p = build(tmp_path, "hsig", fn, (2, 32, 3, 17))
    check(ctx, p, (3 * RNG.standard_normal((2, 32, 3, 17))).astype(np.float32))


def test_linear_silu_and_inexact_weights(ctx, tmp_path):
    def fn(g, x):
        y = g.add("MatMul", [x, w(g, (120, 240), 120)])
        y = g.add("Add", [y, g.init("lb", (RNG.standard_normal(240) * 0.1).astype(np.float32))])
        s = g.add("Sigmoid", [y])
        y = g.add("Mul", [y, s])
        return g.add("MatMul", [y, w(g, (240, 50), 240, exact=False)])
    p = build(tmp_path, "lin", fn, (3, 37, 120))
    check(ctx, p, RNG.standard_normal((3, 37, 120)).astype(np.float32))


def test_layer_norm_and_attention(ctx, tmp_path):
    def fn(g, x):
        b = synth_pp._B("t", 5)
        b.g = g
        return synth_pp._svtr_block(b, x)
    p = build(tmp_path, "svtr", fn, (2, 23, 120))
    check(ctx, p, RNG.standard_normal((2, 23, 120)).astype(np.float32))


def test_pools_resize_convt_concat(ctx, tmp_path):
    def fn(g, x):
        a = g.add("AveragePool", [x], kernel_shape=[3, 3], strides=[2, 2], pads=[1, 1, 1, 1])
        m = g.add("MaxPool", [x], kernel_shape=[3, 3], strides=[2, 2], pads=[1, 1, 1, 1])
        y = g.add("Concat", [a, m], axis=1)
        y = g.add("Resize", [y, "", g.init("sc", np.array([1, 1, 2, 2], np.float32))], mode="nearest",
                  coordinate_transformation_mode="asymmetric", nearest_mode="floor")
        t = g.add("ConvTranspose", [y, w(g, (12, 5, 2, 2), 12), g.init("tb", np.full(5, 0.05, np.float32))],
                  kernel_shape=[2, 2], strides=[2, 2])
        t = g.add("Sigmoid", [t])
        r = g.add("ReduceMean", [t], axes=[2, 3], keepdims=0)
        return g.add("Concat", [r, g.add("Sqrt", [g.add("Mul", [r, r])])], axis=1)
    p = build(tmp_path, "prc", fn, (2, 6, 9, 10))
    check(ctx, p, RNG.standard_normal((2, 6, 9, 10)).astype(np.float32))


def test_binary_broadcast_and_shape_ops(ctx, tmp_path):
    def fn(g, x):
        sh = g.add("Shape", [x])
        nt = g.add("Gather", [sh, ints(g, [0, 1])], axis=0)
        s5 = g.add("Concat", [nt, ints(g, [2, 3])], axis=0)
        y = g.add("Reshape", [x, s5])                       # [2, 5, 2, 3]
        y = g.add("Transpose", [y], perm=[0, 2, 1, 3])      # [2, 2, 5, 3]
        z = g.add("Sub", [y, g.init("row", RNG.standard_normal(3).astype(np.float32))])
        z = g.add("Div", [z, g.init("col", (RNG.uniform(1, 2, (1, 2, 5, 1))).astype(np.float32))])
        z = g.add("Pow", [z, const(g, 2.0)])
        z = g.add("Slice", [z, ints(g, [1, 0]), ints(g, [4, 2]), ints(g, [2, 3])])
        return g.add("Unsqueeze", [g.add("Squeeze", [g.add("Unsqueeze", [z, ints(g, [0])]), ints(g, [0])]), ints(g, [1])])
    p = build(tmp_path, "bin", fn, (2, 5, 6))
    check(ctx, p, RNG.standard_normal((2, 5, 6)).astype(np.float32))


def test_fusions_across_unrelated_nodes_and_operand_orders(ctx, tmp_path):
    # Chains the plan matches over def-use edges rather than node order: a bias Add given first
    # and placed after an unrelated node, a residual produced after the conv, the LayerNorm's
    # gamma Mul with its operands swapped and an unrelated node inside the chain, GELU with its
    # constants first. Each runs fused and must equal the unfused oracle.
    def fn(g, x):
        c = conv(g, x, 8, 16, bias=False)
        side = g.add("Relu", [x])
        y = g.add("Add", [g.init("b0", (RNG.standard_normal((1, 16, 1, 1)) * 0.1).astype(np.float32)), c])
        h = g.add("Erf", [g.add("Div", [y, const(g, 1.4142135)])])
        y = g.add("Mul", [const(g, 0.5), g.add("Mul", [g.add("Add", [const(g, 1.0), h]), y])])
        y = g.add("Add", [conv(g, side, 8, 16), y])
        t = g.add("Reshape", [y, ints(g, [2, 16, -1])])
        m = g.add("ReduceMean", [t], axes=[-1])
        d = g.add("Sub", [t, m])
        v = g.add("ReduceMean", [g.add("Pow", [d, const(g, 2.0)])], axes=[-1])
        other = g.add("Sigmoid", [t])
        n = g.add("Div", [d, g.add("Sqrt", [g.add("Add", [const(g, 1e-5), v])])])
        width = 11 * 13
        n = g.add("Mul", [g.init("gm", RNG.uniform(0.5, 1.5, width).astype(np.float32)), n])
        n = g.add("Add", [n, g.init("bt", RNG.uniform(-.1, .1, width).astype(np.float32))])
        return g.add("Add", [n, other])
    p = build(tmp_path, "defuse", fn, (2, 8, 11, 13))
    import ocrhip
    kinds = [line.split()[0] for line in ocrhip.nd_plan(p)]
    assert kinds.count("layer_norm") == 1 and any("act=gelu" in line and "residual" in line
                                                  for line in ocrhip.nd_plan(p))
    check(ctx, p, RNG.standard_normal((2, 8, 11, 13)).astype(np.float32))


# ---- the N-D convolution and row-GEMM kernels at the PP-OCR shapes --------------------------------
@pytest.mark.parametrize("shape,stride,k", [((2, 32, 24, 70), (1, 1), 3), ((2, 64, 24, 70), (2, 2), 3),
                                            ((3, 128, 12, 37), (2, 1), 3), ((1, 16, 9, 8), (1, 2), 3),
                                            ((2, 24, 13, 29), (2, 2), 5)])
def test_depthwise_shapes(ctx, tmp_path, shape, stride, k):
    c = shape[1]
    p = build(tmp_path, "dw", lambda g, x: g.add("Relu", [bn(g, conv(g, x, c, c, k=k, stride=stride, group=c,
                                                                       bias=False), c)]), shape)
    check(ctx, p, RNG.standard_normal(shape).astype(np.float32))


@pytest.mark.parametrize("cin,cout,h,wd,exact", [(32, 64, 24, 73, True), (64, 128, 12, 37, False),
                                                  (256, 256, 3, 109, True), (120, 256, 1, 61, True),
                                                  (30, 20, 5, 7, True), (128, 32, 1, 1, False)])
def test_1x1_nchw_shapes(ctx, tmp_path, cin, cout, h, wd, exact):
    shape = (3, cin, h, wd)
    p = build(tmp_path, "pw", lambda g, x: g.add("Relu", [bn(g, conv(g, x, cin, cout, k=1, bias=False, exact=exact),
                                                               cout)]), shape)
    check(ctx, p, RNG.standard_normal(shape).astype(np.float32))


@pytest.mark.parametrize("n,cin,cout,h,wd,exact", [(4, 256, 32, 1, 109, True), (3, 512, 32, 1, 61, False),
                                                    (2, 64, 16, 20, 45, True), (2, 40, 24, 7, 130, False),
                                                    (16, 64, 64, 1, 9, True), (2, 960, 64, 1, 49, True),
                                                    (1, 480, 60, 1, 120, False), (5, 960, 48, 1, 37, False)])
def test_3x3_nchw_shapes(ctx, tmp_path, n, cin, cout, h, wd, exact):
    # One-row inputs (the SVTR neck's convs: two of the three kernel rows read padding only, and
    # few tiles make the wavefronts of a workgroup share the K steps, up to 16 of them for a long
    # K: 960 -> 64 and 960 -> 48) and two-dimensional ones.
    shape = (n, cin, h, wd)
    p = build(tmp_path, "c3", lambda g, x: g.add("Relu", [conv(g, x, cin, cout, k=3, exact=exact)]), shape)
    check(ctx, p, RNG.standard_normal(shape).astype(np.float32))


@pytest.mark.parametrize("n,cin,cout,wd,exact", [(2, 1024, 64, 40, True), (3, 1024, 32, 21, False),
                                                 (1, 1200, 16, 300, True)])
def test_1x1_nchw_long_k(ctx, tmp_path, n, cin, cout, wd, exact):
    # 1 x 1 convs with a long K over few pixels: the K steps shared by up to 16 wavefronts of a
    # workgroup, their partial sums added in a fixed order.
    import ocrhip
    shape = (n, cin, 1, wd)
    p = build(tmp_path, "c1k", lambda g, x: conv(g, x, cin, cout, k=1, exact=exact), shape)
    x = RNG.standard_normal(shape).astype(np.float32)
    got, _ = check(ctx, p, x)
    np.testing.assert_array_equal(ocrhip.NdGraph(ctx, p).run(x), got)  # the same bits on a rerun


def test_se_gate_and_gelu_residual_at_pp_shapes(ctx, tmp_path):
    def fn(g, x):
        se = g.add("GlobalAveragePool", [x])
        se = g.add("Relu", [conv(g, se, 128, 32, k=1)])
        se = g.add("HardSigmoid", [conv(g, se, 32, 128, k=1)], alpha=0.2, beta=0.5)
        y = g.add("Relu", [conv(g, g.add("Mul", [x, se]), 128, 256, k=1)])
        z = conv(g, y, 256, 256, k=1)
        d = g.add("Div", [z, const(g, np.float32(np.sqrt(2.0)))])
        m = g.add("Mul", [z, g.add("Add", [g.add("Erf", [d]), const(g, 1.0)])])
        return g.add("Add", [g.add("Mul", [m, const(g, 0.5)]), y])
    p = build(tmp_path, "se2", fn, (3, 128, 6, 45))
    check(ctx, p, RNG.standard_normal((3, 128, 6, 45)).astype(np.float32))


@pytest.mark.parametrize("cin,cout,shape,stride", [(3, 32, (2, 3, 48, 97), (2, 2)), (1, 16, (3, 1, 21, 40), (1, 1)),
                                                    (3, 48, (1, 3, 33, 35), (2, 1))])
def test_stem_convs(ctx, tmp_path, cin, cout, shape, stride):
    p = build(tmp_path, "stem", lambda g, x: g.add("Relu", [bn(g, conv(g, x, cin, cout, stride=stride, bias=False),
                                                                 cout)]), shape)
    check(ctx, p, RNG.standard_normal(shape).astype(np.float32))


@pytest.mark.parametrize("shape,k,n,exact", [((16, 109, 120), 120, 360, True), ((64, 200, 120), 120, 240, False),
                                             ((2, 21, 30), 30, 7, True), ((5, 33, 240), 240, 120, True)])
def test_linear_row_gemm_shapes(ctx, tmp_path, shape, k, n, exact):
    def fn(g, x):
        y = g.add("MatMul", [x, w(g, (k, n), k, exact=exact)])
        return g.add("Add", [y, g.init("lb", (RNG.standard_normal(n) * 0.1).astype(np.float32))])
    p = build(tmp_path, "rows", fn, shape)
    check(ctx, p, RNG.standard_normal(shape).astype(np.float32))


@pytest.mark.parametrize("rows,k,n,exact", [(3305, 120, 1301, True), (4100, 200, 1100, False), (3296, 64, 1344, True)])
def test_linear_many_columns(ctx, tmp_path, rows, k, n, exact):
    # Enough rows and columns for ranges of column blocks a wavefront; rows, K and N that end inside
    # a tile, chunk and block.
    def fn(g, x):
        y = g.add("MatMul", [x, w(g, (k, n), k, exact=exact)])
        return g.add("Add", [y, g.init("lb", (RNG.standard_normal(n) * 0.1).astype(np.float32))])
    p = build(tmp_path, "wide", fn, (1, rows, k))
    x = RNG.standard_normal((1, rows, k)).astype(np.float32)
    assert ran(["nd_rows_wide"], lambda: check(ctx, p, x)) == {"nd_rows_wide": 1}


@pytest.mark.parametrize("k,n,exact", [(120, 200, True), (256, 300, False), (64, 1000, True)])
def test_head_argmax_first_index_on_ties(ctx, tmp_path, k, n, exact):
    """The fused head: classes come in pairs with the same weights and bias, so every row's
    maximum is a tie; the first index of the pair must win (nd.rs:383), as in the oracle's
    logits."""
    import ocrhip

    def fn(g, x):
        a = RNG.standard_normal((k, n // 2)).astype(np.float32) * np.float32(np.sqrt(2 / k))
        a = f16x(a) if exact else a
        wt = np.repeat(a, 2, axis=1)
        bias = np.repeat((RNG.standard_normal(n // 2) * 0.1).astype(np.float32), 2)
        y = g.add("MatMul", [x, g.init("hw", wt)])
        y = g.add("Add", [y, g.init("hb", bias)])
        return g.add("Softmax", [y], axis=-1)
    shape = (3, 41, k)
    p = build(tmp_path, "head", fn, shape)
    x = RNG.standard_normal(shape).astype(np.float32)
    head = ocrhip.NdGraph(ctx, p, stop_before_softmax=True)
    got = head.argmax(x)
    probs, _ = og.run(onnx_read.load(p), x)
    want = np.argmax(probs, axis=-1)  # equal logits give equal probabilities: the first index
    assert np.all(want % 2 == 0)
    assert np.all(got % 2 == 0), "a tie went to the second index"
    assert np.array_equal(got, want)
    assert np.array_equal(got, np.argmax(head.run(x), axis=-1))


@pytest.mark.parametrize("c,h,wd,stride,k", [(2, 3, 1, (1, 1), 3), (3, 4, 3, (1, 1), 3), (3, 5, 4, (2, 2), 3), (3, 5, 5, (1, 1), 3),
                                             (2, 6, 6, (2, 2), 3), (2, 7, 7, (1, 2), 3), (2, 5, 9, (2, 2), 5), (2, 5, 4, (1, 1), 5),
                                             (2, 5, 6, (2, 1), 5)])
def test_depthwise_row_ends(ctx, tmp_path, c, h, wd, stride, k):
    # Rows that end inside or before a 16-byte load, at every shift.
    p = build(tmp_path, "dwe", lambda g, x: conv(g, x, c, c, k=k, stride=stride, group=c, exact=False), (2, c, h, wd))
    x = RNG.standard_normal((2, c, h, wd)).astype(np.float32)
    assert ran(["nd_conv_dw", "nd_conv_dw_wide"], lambda: check(ctx, p, x)) == {"nd_conv_dw": 1, "nd_conv_dw_wide": int(wd >= 4)}


@pytest.mark.parametrize("cin,cout,h,wd,s,form", [
    (6, 5, 7, 9, 2, "nd_convt_1"), (4, 3, 16, 17, 2, "nd_convt_1"), (3, 6, 5, 5, 1, "nd_convt_1"), (4, 2, 3, 3, 3, "nd_convt_1"),
    (6, 5, 130, 252, 2, "nd_convt_4"), (6, 5, 127, 256, 2, "nd_convt_1"), (3, 6, 257, 131, 1, "nd_convt_4"), (4, 2, 300, 300, 3, "nd_convt_1")])
def test_conv_transpose_channel_blocks(ctx, tmp_path, cin, cout, h, wd, s, form):
    # Output channels that do not fill a thread's four, and planes that end inside a workgroup.
    p = build(tmp_path, "ctb", lambda g, x: g.add("ConvTranspose", [x, w(g, (cin, cout, s, s), cin, exact=False),
                                                                     g.init("tb", np.full(cout, 0.1, np.float32))],
                                                  kernel_shape=[s, s], strides=[s, s]), (2, cin, h, wd))
    x = RNG.standard_normal((2, cin, h, wd)).astype(np.float32)
    assert ran([form], lambda: check(ctx, p, x)) == {form: 1}


@pytest.mark.parametrize("h,wd", [(1, 1), (3, 31), (2, 32), (5, 33), (4, 64), (3, 255), (2, 257), (7, 736)])
def test_threshold_bits_widths(ctx, h, wd):
    # One bit a pixel, rows of whole words: the bits past a row's end are zero, equal is not above.
    import ocrhip
    prob = RNG.choice(np.array([0.0, 0.3, np.nextafter(np.float32(0.3), np.float32(1)), 1.0], np.float32), (h, wd))
    got = ocrhip.db_threshold(ctx, prob, 0.3)
    on = np.zeros((h, (wd + 31) // 32 * 32), np.uint8)
    on[:, :wd] = prob > np.float32(0.3)
    want = np.packbits(on, axis=1, bitorder="little").view(np.uint32)
    assert np.array_equal(np.asarray(got, np.uint32).reshape(want.shape), want)


@pytest.mark.parametrize("cin,cout,k,s,act", [(16, 16, 2, 2, "Relu"), (16, 1, 2, 2, "Sigmoid"), (8, 5, 3, 3, "Relu"),
                                             (6, 4, 3, 2, "Sigmoid"), (5, 7, 4, 4, None)])
def test_conv_transpose_nchw_shapes(ctx, tmp_path, cin, cout, k, s, act):
    # kernel = stride (each input pixel alone makes its s x s outputs) and an overlapping one
    def fn(g, x):
        y = g.add("ConvTranspose", [x, w(g, (cin, cout, k, k), cin), g.init("tb", (RNG.standard_normal(cout) * 0.1)
                                                                          .astype(np.float32))],
                  kernel_shape=[k, k], strides=[s, s])
        return g.add(act, [y]) if act else y
    shape = (2, cin, 23, 37)
    p = build(tmp_path, "convt", fn, shape)
    check(ctx, p, RNG.standard_normal(shape).astype(np.float32))


def _attention(g, x, dim, heads):
    return _attention_of(g, g.add("MatMul", [x, w(g, (dim, 3 * dim), dim)]), dim, heads)


def _attention_of(g, qkv, dim, heads):
    hd = dim // heads
    t5 = g.add("Transpose", [g.add("Reshape", [qkv, ints(g, [0, 0, 3, heads, hd])])], perm=[2, 0, 3, 1, 4])
    parts = [g.add("Squeeze", [g.add("Slice", [t5, ints(g, [i]), ints(g, [i + 1]), ints(g, [0])]), ints(g, [0])])
             for i in range(3)]
    q = g.add("Mul", [parts[0], const(g, np.float32(hd ** -0.5))])
    att = g.add("Softmax", [g.add("MatMul", [q, g.add("Transpose", [parts[1]], perm=[0, 1, 3, 2])])], axis=-1)
    o = g.add("Transpose", [g.add("MatMul", [att, parts[2]])], perm=[0, 2, 1, 3])
    return g.add("Reshape", [o, ints(g, [0, 0, dim])])


@pytest.mark.parametrize("n,t,dim,heads", [(3, 37, 120, 8), (2, 300, 120, 8), (2, 77, 64, 2), (1, 150, 128, 2),
                                           (4, 1, 48, 4)])
def test_fused_attention_shapes(ctx, tmp_path, n, t, dim, heads):
    # Heads of 15, 32 and 64 values; 300 and 150 keys take several LDS tiles (the running softmax
    # rescaled between them); one query alone.
    import ocrhip
    p = build(tmp_path, "attn", lambda g, x: _attention(g, x, dim, heads), (n, t, dim))
    assert any(line.startswith("attention") for line in ocrhip.nd_plan(p))
    x = RNG.standard_normal((n, t, dim)).astype(np.float32)
    calls = ran(["nd_attention", "nd_attention_mfma"], lambda: check(ctx, p, x))
    assert calls == {"nd_attention": 1, "nd_attention_mfma": int(4 <= dim // heads <= 16)}


@pytest.mark.parametrize("d,form", [(1, "nd_attention_16"), (2, "nd_attention_16"), (3, "nd_attention_16"),
                                    (4, "nd_attention_mfma"), (16, "nd_attention_mfma"), (17, "nd_attention_32"),
                                    (32, "nd_attention_32"), (33, "nd_attention_64")])
def test_attention_head_sizes(ctx, tmp_path, d, form):
    # Each kernel at the ends of its head sizes: the smallest vectors that hold a head.
    p = build(tmp_path, "hs", lambda g, x: _attention(g, x, 3 * d, 3), (2, 45, 3 * d))
    x = RNG.standard_normal((2, 45, 3 * d)).astype(np.float32)
    assert ran([form], lambda: check(ctx, p, x)) == {form: 1}


@pytest.mark.parametrize("proj", [False, True])
@pytest.mark.parametrize("t,d,heads", [(77, 15, 3), (33, 4, 8), (70, 6, 2), (40, 3, 4), (70, 16, 1)])
def test_attention_infinities(ctx, tmp_path, t, d, heads, proj):
    # Keys that a query scores at -inf weigh nothing, wherever they lie: all of the first 37 keys or
    # but one, the score's infinity in the head's first value or in one of its last (which the
    # kernels' loads may hold twice). An infinite value of the last key is an infinite output, not
    # NaN (without the projection, whose float16 parts hold no infinities).
    dim = heads * d
    x = RNG.standard_normal((2, t, 3, heads, d)).astype(np.float32)
    where = (0, d - 1, max(0, d - 4))
    for v in where:
        x[:, :, 0, :, v] = np.abs(x[:, :, 0, :, v]) + np.float32(0.1)
    x[0, :min(37, t - 1), 1, :, where[0]] = -np.inf
    x[1, 5, 1, :, where[1]] = x[1, 7, 1, :, where[2]] = -np.inf
    if not proj:
        x[1, t - 1, 2, :, d // 2] = np.inf
    x = x.reshape(2, t, 3 * dim)

    def fn(g, xi):
        y = _attention_of(g, xi, dim, heads)
        return _linear(g, g.add("Relu", [_linear(g, y, dim, 20, True)]), 20, 8, True) if proj else y
    p = build(tmp_path, "inf", fn, x.shape)
    import ocrhip
    form = "nd_attention_16" if d < 4 else "nd_attention_proj" if proj else "nd_attention_mfma"
    got = []
    assert ran([form], lambda: got.append(ocrhip.NdGraph(ctx, p).run(x))) == {form: 1}
    want, _ = og.run(onnx_read.load(p), x)
    assert not np.isnan(want).any() and np.isinf(want).any() == (not proj)
    assert np.array_equal(np.isinf(got[0]), np.isinf(want)), "infinities"
    fin = np.isfinite(want)
    assert (np.abs(got[0][fin] - want[fin]) <= 1e-4 * (1 + np.abs(want[fin]))).all()


@pytest.mark.parametrize("heads,d", [(4, 3), (2, 24), (20, 16)])
def test_attention_and_projection_apart(ctx, tmp_path, heads, d):
    # Sizes that the joined kernel does not take: attention, then the projection as any Linear runs.
    dim = heads * d
    p = build(tmp_path, "ap", lambda g, x: g.add("Relu", [_linear(g, _attention(g, x, dim, heads), dim, 40, False)]), (2, 37, dim))
    x = RNG.standard_normal((2, 37, dim)).astype(np.float32)
    calls = ran(["nd_attention", "nd_attention_proj", "nd_gemm_rows"], lambda: check(ctx, p, x))
    assert calls == {"nd_attention": 1, "nd_attention_proj": 0, "nd_gemm_rows": 2}


@pytest.mark.parametrize("kind,m,hidden,n,joined", [
    ("norm", 33, 0, 720, True), ("norm", 33, 0, 736, False), ("norm", 800, 0, 800, True), ("norm", 799, 0, 800, False),
    ("norm", 13200, 0, 56, True), ("norm", 13201, 0, 56, False), ("norm", 24100, 0, 200, True),
    ("mlp", 8000, 16, 20, True), ("mlp", 8001, 16, 20, False), ("normmlp", 20, 64, 750, False),
    ("attention", 74, 0, 700, True), ("attention", 74, 0, 740, False)])
def test_joined_steps_where_they_pay(ctx, tmp_path, kind, m, hidden, n, joined):
    # Both sides of the lines up to which a step joined into one launch is the faster, with a residual
    # and inexact weights in the second product.
    k = 120
    def fn(g, x):
        if kind == "attention":
            y = _attention_of(g, x, k, 8)
        else:
            y = _layer_norm(g, x, k) if "norm" in kind else x
        if hidden:
            y = _linear(g, y, k, hidden, True, act=True)
        y = _linear(g, y, hidden or k, n, not hidden)
        if n <= 200:
            y = g.add("Add", [y, _linear(g, x, 3 * k if kind == "attention" else k, n, True)])
        return g.add("Relu", [y])
    shape = (2, m // 2, 3 * k) if kind == "attention" else (1, m, k)
    p = build(tmp_path, "pays", fn, shape)
    x = RNG.standard_normal(shape).astype(np.float32)
    form = {"norm": "nd_rows_norm", "attention": "nd_attention_proj"}.get(kind, "nd_mlp")
    norms = int("norm" in kind)
    calls = ran([form, "nd_layer_norm"], lambda: check(ctx, p, x))
    assert calls == {form: int(joined), "nd_layer_norm": 0 if joined else norms}


def _pool2(g, x):
    return g.add("MaxPool", [x], kernel_shape=[2, 2], strides=[2, 2])


def _up(g, x, f):
    sc = g.init(g.fresh("sc"), np.array([1, 1, f, f], np.float32))
    return g.add("Resize", [x, "", sc], mode="nearest", coordinate_transformation_mode="asymmetric", nearest_mode="floor")


@pytest.mark.parametrize("n,cin,cout,h,w,exact,tiled", [
    (3, 20, 16, 41, 101, True, 0), (1, 64, 40, 64, 289, False, 2), (1, 64, 40, 64, 249, False, 0), (2, 33, 64, 120, 90, True, 0), (1, 3, 70, 96, 200, True, 2),
    (3, 20, 16, 81, 101, True, 2), (1, 64, 40, 121, 417, False, 2), (2, 130, 64, 120, 138, True, 1), (1, 100, 16, 96, 174, False, 1),
    (2, 36, 30, 105, 155, False, 2), (4, 64, 64, 60, 46, True, 0)])
def test_3x3_nchw_many_rows(ctx, tmp_path, n, cin, cout, h, w, exact, tiled):
    # Images of many rows: tiles of 8 x 32 pixels with a part of a tile left on both sides, channel
    # counts that end inside a chunk or block, with a residual. From the sizes on at which tiles are
    # the faster, by block, channels and row length (tiled: how many of the two convs).
    def fn(g, x):
        y = g.add("Relu", [bn(g, conv(g, x, cin, cout, exact=exact, bias=False), cout)])
        return g.add("Add", [g.add("Relu", [conv(g, y, cout, cout)]), y])
    p = build(tmp_path, "c3r", fn, (n, cin, h, w))
    x = RNG.standard_normal((n, cin, h, w)).astype(np.float32)
    assert ran(["nd_conv_tile"], lambda: check(ctx, p, x)) == {"nd_conv_tile": tiled}


@pytest.mark.parametrize("n,c,h,w,cout,inplace", [(4, 16, 64, 96, 16, True), (1, 16, 16, 24, 16, False), (2, 8, 88, 160, 40, True),
                                                  (2, 12, 64, 96, 16, False), (4, 32, 32, 104, 32, True)])
def test_conv_of_upscaled_parts(ctx, tmp_path, n, c, h, w, cout, inplace):
    # What a Concat of Resizes would write is read from the parts: by the 3 x 3 conv on tiles, or
    # written out after all (few tiles, a part of 12 channels). A Resize is also a 1 x 1 and a
    # 3 x 3 conv's residual, and one is read by an op that is no conv.
    def fn(g, x):
        p1 = _pool2(g, x)
        p2 = _pool2(g, p1)
        u1 = _up(g, p1, 2.0)
        cat = g.add("Concat", [_up(g, p2, 4.0), u1, x], axis=1)
        y = g.add("Relu", [conv(g, cat, 3 * c, cout)])
        a = g.add("Add", [conv(g, y, cout, c, k=1), u1])
        b = g.add("Add", [conv(g, a, c, c), _up(g, p1, 2.0)])
        return g.add("Add", [b, g.add("Relu", [_up(g, p2, 4.0)])])
    p = build(tmp_path, "parts", fn, (n, c, h, w))
    x = RNG.standard_normal((n, c, h, w)).astype(np.float32)
    calls = ran(["nd_copy", "nd_resize"], lambda: check(ctx, p, x))
    assert calls == {"nd_copy": 0 if inplace else 3, "nd_resize": 1 if inplace else 3}


def test_parts_written_out_once(ctx, tmp_path):
    # Readers that cannot take parts share one written-out value: a Resize of two 1 x 1 convs, which
    # a Concat of two 3 x 3 convs (few pixels) holds as well, and a Concat whose first part does not
    # end with a chunk, of two 1 x 1 convs.
    def fn(g, x):
        a = g.add("Relu", [conv(g, x, 8, 24, k=1)])
        u = _up(g, _pool2(g, a), 2.0)
        v = _up(g, _pool2(g, _pool2(g, a)), 4.0)
        y = [conv(g, u, 24, 16, k=1), conv(g, u, 24, 16, k=1)]
        cat = g.add("Concat", [u, v], axis=1)
        y += [conv(g, cat, 48, 16), conv(g, cat, 48, 16)]
        two = g.add("Concat", [a, g.add("Relu", [conv(g, x, 8, 9, k=1)])], axis=1)
        y += [conv(g, two, 33, 16, k=1), conv(g, two, 33, 16, k=1)]
        out = y[0]
        for v in y[1:]:
            out = g.add("Add", [g.add("Relu", [out]), g.add("Sigmoid", [v])])
        return out
    p = build(tmp_path, "once", fn, (1, 8, 12, 20))
    x = RNG.standard_normal((1, 8, 12, 20)).astype(np.float32)
    calls = ran(["nd_resize", "nd_copy", "nd_conv_tile"], lambda: check(ctx, p, x))
    assert calls == {"nd_resize": 2, "nd_copy": 4, "nd_conv_tile": 0}


@pytest.mark.parametrize("n,c1,c2,h,w,k", [(2, 256, 256, 1, 109, 3), (1, 32, 40, 5, 61, 1), (3, 64, 16, 9, 30, 3), (2, 24, 40, 6, 50, 1)])
def test_conv_of_two_tensors(ctx, tmp_path, n, c1, c2, h, w, k):
    # A conv over a Concat of two tensors reads both where they lie (the first of a multiple of 32
    # channels; the last case is written out).
    def fn(g, x):
        a = g.add("Relu", [conv(g, x, 16, c1, k=1)])
        b = g.add("Relu", [conv(g, x, 16, c2, k=1)])
        return g.add("Relu", [conv(g, g.add("Concat", [a, b], axis=1), c1 + c2, 40, k=k)])
    p = build(tmp_path, "two", fn, (n, 16, h, w))
    x = RNG.standard_normal((n, 16, h, w)).astype(np.float32)
    assert ran(["nd_copy"], lambda: check(ctx, p, x)) == {"nd_copy": 2 if c1 % 32 else 0}


@pytest.mark.parametrize("k", [1, 3])
@pytest.mark.parametrize("scale,up", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("n,c1,c2,h,w", [(2, 32, 40, 6, 50), (1, 64, 8, 2, 26)])
def test_conv_of_two_tensors_scaled(ctx, tmp_path, n, c1, c2, h, w, k, scale, up, exact):
    # The same with an input scale, whose channels run on over both tensors (the second ends inside
    # a chunk), and with an upscaled residual, read where they lie.
    c, cout = c1 + c2, 24
    def fn(g, x):
        a = g.add("Relu", [conv(g, x, 16, c1, k=1)])
        b = g.add("Relu", [conv(g, x, 16, c2, k=1)])
        y = g.add("Concat", [a, b], axis=1)
        if scale:
            se = conv(g, g.add("GlobalAveragePool", [x]), 16, c, k=1)
            y = g.add("Mul", [y, g.add("HardSigmoid", [se], alpha=0.2, beta=0.5)])
        y = conv(g, y, c, cout, k=k, exact=exact)
        if up:
            y = g.add("Add", [y, _up(g, _pool2(g, conv(g, x, 16, cout, k=1)), 2.0)])
        return g.add("Sigmoid", [y])
    p = build(tmp_path, "twos", fn, (n, 16, h, w))
    x = RNG.standard_normal((n, 16, h, w)).astype(np.float32)
    assert ran(["nd_copy", "nd_resize"], lambda: check(ctx, p, x)) == {"nd_copy": 0, "nd_resize": 0}


@pytest.mark.parametrize("cin,cout,h,w,exact", [(7, 20, 3, 5, True), (64, 16, 9, 31, False), (100, 70, 12, 40, True),
                                                (250, 64, 5, 33, True), (128, 256, 6, 218, False)])
def test_1x1_nchw_channel_edges(ctx, tmp_path, cin, cout, h, w, exact):
    # 1 x 1 convs whose channels end inside a chunk and take one to two batches of chunks, with a
    # GELU and a residual.
    def fn(g, x):
        y = conv(g, x, cin, cout, k=1, exact=exact)
        return g.add("Add", [g.add("Relu", [conv(g, y, cout, cout, k=1, exact=exact)]), y])
    p = build(tmp_path, "c1e", fn, (2, cin, h, w))
    x = RNG.standard_normal((2, cin, h, w)).astype(np.float32)
    assert ran(["nd_conv_px"], lambda: check(ctx, p, x)) == {"nd_conv_px": 2}


def _layer_norm(g, x, k):
    b = synth_pp._B("ln", 3)
    b.g = g
    b.rng = RNG
    return b.layer_norm(x, k)


def _linear(g, x, k, n, exact, act=None):
    y = g.add("MatMul", [x, w(g, (k, n), k, exact)])
    y = g.add("Add", [y, g.init(g.fresh("lb"), (RNG.standard_normal(n) * 0.1).astype(np.float32))])
    return g.add("Mul", [y, g.add("Sigmoid", [y])]) if act else y


@pytest.mark.parametrize("n,t,dim,heads,hidden,exact", [(1, 1, 120, 8, 240, True), (2, 17, 120, 8, 256, False),
                                                        (3, 109, 48, 12, 33, True), (2, 200, 128, 8, 100, False),
                                                        (1, 33, 36, 9, 16, True), (2, 40, 132, 11, 300, True)])
def test_transformer_block_shapes(ctx, tmp_path, n, t, dim, heads, hidden, exact):
    # A block whose parts run joined (normalised QKV, attention with its projection, the MLP): rows
    # and keys at the edges of 16 and 32, heads of 4, 15 and 16 values and more heads than a
    # workgroup has wavefronts, hidden sizes up to the joined kernel's most; the last case is too
    # wide for it and runs in parts.
    def fn(g, x):
        x = g.add("Add", [x, _linear(g, _attention(g, _layer_norm(g, x, dim), dim, heads), dim, dim, exact)])
        y = _linear(g, _layer_norm(g, x, dim), dim, hidden, exact, act=True)
        x = g.add("Add", [x, _linear(g, y, hidden, dim, exact)])
        # The graph's last step stays on its own. (It was a square root: that takes an error e of a value
        # near zero to sqrt(e), 2e-8 to 1.4e-4, past check's bound for some draws.)
        return g.add("Relu", [x])
    p = build(tmp_path, "block", fn, (n, t, dim))
    x = RNG.standard_normal((n, t, dim)).astype(np.float32)
    calls = ran(["nd_layer_norm", "nd_rows_norm", "nd_mlp", "nd_attention_proj"], lambda: check(ctx, p, x))
    fits = dim <= 128
    assert calls == {"nd_layer_norm": 0 if fits else 2, "nd_rows_norm": int(fits), "nd_mlp": int(fits), "nd_attention_proj": 1}


def test_output_memory(ctx, tmp_path):
    # The last step writes the caller's memory; where that is unaligned or the input itself, the
    # output still arrives whole.
    import ctypes
    import ocrhip
    p = build(tmp_path, "om", lambda g, x: g.add("MatMul", [x, w(g, (64, 64), 64)]), (3, 5, 64))
    x = RNG.standard_normal((3, 5, 64)).astype(np.float32)
    graph, lib = ocrhip.NdGraph(ctx, p), ocrhip.lib()
    want = graph.run(x)
    shape = (ctypes.c_int64 * 3)(*x.shape)
    buf = ocrhip.DeviceBuffer(ctx, 4 * x.size + 8192)
    for off_in, off_out in ((0, 4096), (0, 4100), (0, 0), (16, 20)):
        assert lib.ocr_memcpy_h2d(ctx.handle, buf.ptr + off_in, x.ctypes.data, x.nbytes) == 0
        assert lib.ocr_nd_run_device(graph.handle, buf.ptr + off_in, shape, 3, buf.ptr + off_out) == 0
        got = np.empty_like(want)
        assert lib.ocr_memcpy_d2h(ctx.handle, got.ctypes.data, buf.ptr + off_out, got.nbytes) == 0
        assert np.array_equal(got, want), (off_in, off_out)
    buf.free()


def test_unsupported_and_bad_shapes_raise(ctx, tmp_path):
    import ocrhip
    p = build(tmp_path, "bad", lambda g, x: g.add("Tanh", [x]), (1, 4))
    g = ocrhip.NdGraph(ctx, p)
    with pytest.raises(ocrhip.OcrError, match="unsupported op Tanh"):
        g.run(np.zeros((1, 4), np.float32))
    p = build(tmp_path, "c", lambda g, x: conv(g, x, 8, 8), (1, 8, 5, 5))
    with pytest.raises(ocrhip.OcrError, match="channels"):
        ocrhip.NdGraph(ctx, p).run(np.zeros((1, 6, 5, 5), np.float32))


# ---- the PP-OCRv6-architecture models ------------------------------------------------------------
@pytest.fixture(scope="module")
def pp_rec_path():
    return synth_pp.model_path("rec")


@pytest.fixture(scope="module")
def pp_lines():
    return synth_pp.batch_lines(synth_pp.rec_lines(36))


def test_pp_recognition_config4(ctx, pp_rec_path, pp_lines):
    """36 lines, widths in [160, 960], batches sorted by width (16 a batch): the GPU's softmax
    within 1e-3 of the oracle's and the identical arg-max (the fused head) at every step."""
    import ocrhip
    full = ocrhip.NdGraph(ctx, pp_rec_path)
    head = ocrhip.NdGraph(ctx, pp_rec_path, stop_before_softmax=True)
    model = onnx_read.load(pp_rec_path)
    batches, _ = pp_lines
    steps = 0
    for data, n, wd in batches:
        print(f"pp rec batch n={n} w={wd}", flush=True)
        want, _ = og.run(model, data)
        got = full.run(data)
        assert got.shape == want.shape == (n, wd // 8, synth_pp.PP_CLASSES)
        assert np.abs(got - want).max() <= 1e-3
        best = head.argmax(data)
        want_best = np.argmax(want, axis=-1)  # first index on ties, as nd.rs:383
        assert np.array_equal(best, want_best), f"{int((best != want_best).sum())} steps differ"
        steps += best.size
    assert steps == sum(n * wd // 8 for _, n, wd in batches)


def test_pp_head_argmax_matches_materialised_logits(ctx, pp_rec_path, pp_lines):
    """The fused head arg-max equals the arg-max over the head's own logits on the GPU."""
    import ocrhip
    head = ocrhip.NdGraph(ctx, pp_rec_path, stop_before_softmax=True)
    data, n, wd = pp_lines[0][0]
    logits = head.run(data)
    assert np.array_equal(head.argmax(data), np.argmax(logits, axis=-1))


def test_pp_det_input_matches_oracle(ctx):
    import ocrhip
    from ocrhip import synth
    page = np.ascontiguousarray(synth.page(1)[:1700, :1300])
    got = ocrhip.det_input(ctx, page, synth_pp.DET_MAX_SIDE)
    want = og.det_prep(page, synth_pp.DET_MAX_SIDE)
    assert got.shape == want.shape
    # The same float32 operations in the same order, none fused, on both sides: bit-exact.
    np.testing.assert_array_equal(got, want)


def test_pp_detection_map_and_threshold(ctx):
    """The DB detector on a 960 x 736 input: probabilities within 1e-4 of the oracle; the GPU
    threshold (0.3) bit-exact against the oracle's on the same map."""
    import ocrhip
    path = synth_pp.model_path("det")
    x = RNG.standard_normal((1, 3, 960, 736)).astype(np.float32)
    got, want = check(ctx, path, x)
    assert np.abs(got - want).max() <= 1e-4
    bits = ocrhip.db_threshold(ctx, got[0, 0], 0.3)
    assert np.array_equal(bits, og.threshold_bits(got[0, 0], 0.3))
    band = np.abs(want[0, 0] - 0.3) < 1e-4
    assert np.array_equal((got[0, 0] > 0.3)[~band], (want[0, 0] > 0.3)[~band])
