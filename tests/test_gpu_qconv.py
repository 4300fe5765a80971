"""GPU parity of QLinearConv (ingot_rocm_qlinear_conv and the QLinearConv@10 op).

Bar: bit-exact against the oracle's restatement of the reference
(qlinearConvOp.Run, ops/quant.go:343-706), on the geometries of the
reference's TestQLinearConv (ops/quant_optest_test.go:133-192) and on larger
shapes that take an int8 MFMA GEMM. Every device route runs every case:
INGOT_QCONV_PATH=1 forces the direct kernel, 2 the pixel GEMM, 3 im2col and
the GEMM over its column matrix; 4 the depthwise kernels wherever they hold.
"""

import numpy as np
import pytest

import oracle
from helpers import announce
from ingot_amd import IngotError
from ingot_amd import _lib as L
from test_oracle_qconv import REF_CFGS

pytestmark = pytest.mark.gpu

DT = {np.dtype(np.uint8): L.DT_U8, np.dtype(np.int8): L.DT_I8}


ROUTES = {"auto": "0", "direct": "1", "pixel": "2", "im2col": "3"}


@pytest.fixture(params=list(ROUTES))
def route(request):
    return request.param


@pytest.fixture
def qsess(env_session, route):
    """A session whose QLinearConv route is forced (INGOT_QCONV_PATH, read when the session opens)."""
    return env_session(INGOT_QCONV_PATH=ROUTES[route])


def make_case(rng, n, c, h, w, m, kh, kw, g, x_dtype=np.uint8, zx=120, with_bias=True, per_channel=True):
    if x_dtype == np.uint8:
        x = rng.integers(0, 256, (n, c, h, w), dtype=np.uint8)
    else:
        x = rng.integers(-128, 128, (n, c, h, w), dtype=np.int8)
    wt = rng.integers(-128, 128, (m, c // g, kh, kw), dtype=np.int8)
    bias = (rng.integers(0, 2048, m) - 1024).astype(np.int32) if with_bias else None
    xs, ys = 0.02, 0.4
    wsc = (np.float32(0.01) + np.arange(m, dtype=np.float32) * np.float32(0.003)) if per_channel else \
        np.array([0.013], np.float32)
    # keep outputs inside the requant range for wide reductions
    wsc = (wsc / np.float32(max(1.0, np.sqrt(c // g * kh * kw / 9.0)))).astype(np.float32)
    mult = oracle.qconv_mult(xs, wsc, ys, m)
    return x, zx, wt, bias, mult, xs, wsc, ys


def run_conv(sess, x, zx, wt, bias, mult, zy, y_u8, group=1, strides=(1, 1), dilations=(1, 1), pads=(0, 0, 0, 0)):
    n, c, h, w = x.shape
    m, cg, kh, kw = wt.shape
    oh = oracle.conv_out(h, kh, strides[0], dilations[0], pads[0], pads[2])
    ow = oracle.conv_out(w, kw, strides[1], dilations[1], pads[1], pads[3])
    pw = sess.upload_weight(wt.reshape(m, -1), trans=True, pack_dtype=L.DT_I8)
    dx = sess.to_device(x, DT[x.dtype])
    dm = sess.to_device(np.ascontiguousarray(mult, np.float32))
    db = sess.to_device(bias) if bias is not None else None
    y = sess.empty(L.DT_U8 if y_u8 else L.DT_I8, (n, m, max(oh, 0), max(ow, 0)))
    try:
        sess.qlinear_conv(dx, zx, pw, wt.shape, dm, zy, y, bias=db, group=group, strides=strides,
                          dilations=dilations, pads=pads)
        return y.numpy()
    finally:
        for t in (pw, dx, dm, db, y):
            if t is not None:
                t.free()


@pytest.mark.parametrize("cfg", REF_CFGS, ids=[f"c{i}" for i in range(len(REF_CFGS))])
@pytest.mark.parametrize("x_dtype,zx,y_u8,zy", [(np.uint8, 120, True, 17), (np.int8, -7, False, -3)])
def test_reference_geometries(qsess, route, cfg, x_dtype, zx, y_u8, zy):
    sess = qsess
    n, c, h, w, m, kh, kw, g, sh, sw, pt, pl = cfg
    announce(f"qconv ref cfg {cfg} x={np.dtype(x_dtype).name} route={route}")
    rng = np.random.default_rng(hash(cfg) % 2**32)
    x, zx, wt, bias, mult, *_ = make_case(rng, n, c, h, w, m, kh, kw, g, x_dtype, zx)
    kw_ = dict(group=g, strides=(sh, sw), pads=(pt, pl, pt, pl))
    got = run_conv(sess, x, zx, wt, bias, mult, zy, y_u8, **kw_)
    want = oracle.qlinear_conv(x, zx, wt, bias, mult, zy, y_u8, **kw_)
    np.testing.assert_array_equal(got, want)


# Shapes of the GEMM route: several k-tiles, K off the 128 grid, rows off the
# tile grid, groups with a GEMM each, strides, dilations, asymmetric pads, 1×1.
GEMM_CASES = [
    # n, c, h, w, m, kh, kw, g, strides, dilations, pads
    (1, 64, 28, 28, 64, 3, 3, 1, (1, 1), (1, 1), (1, 1, 1, 1)),
    (2, 32, 17, 13, 48, 3, 3, 1, (2, 2), (2, 2), (2, 0, 1, 3)),
    (1, 32, 15, 15, 64, 3, 3, 2, (1, 1), (1, 1), (1, 1, 1, 1)),
    (2, 256, 14, 14, 128, 1, 1, 1, (1, 1), (1, 1), (0, 0, 0, 0)),
    (1, 3, 33, 31, 32, 7, 7, 1, (2, 2), (1, 1), (3, 3, 3, 3)),
    (3, 48, 9, 10, 96, 5, 3, 3, (1, 2), (1, 1), (2, 1, 2, 1)),
    (1, 130, 6, 5, 20, 1, 2, 1, (1, 1), (1, 1), (0, 0, 0, 1)),
]


@pytest.mark.parametrize("case", GEMM_CASES, ids=[f"g{i}" for i in range(len(GEMM_CASES))])
def test_gemm_shapes(qsess, route, case):
    sess = qsess
    n, c, h, w, m, kh, kw, g, st, dl, pads = case
    if route == "direct" and c * h * w * m * kh * kw // g > 5e7:
        pytest.skip("the direct route is covered on the smaller cases")
    announce(f"qconv gemm case {case} route={route}")
    rng = np.random.default_rng(sum(case[:7]))
    for x_dtype, zx, y_u8, zy, with_bias, per_ch in [(np.uint8, 131, True, 9, True, True),
                                                      (np.int8, 4, False, 0, False, False)]:
        x, zx, wt, bias, mult, *_ = make_case(rng, n, c, h, w, m, kh, kw, g, x_dtype, zx, with_bias, per_ch)
        kw_ = dict(group=g, strides=st, dilations=dl, pads=pads)
        got = run_conv(sess, x, zx, wt, bias, mult, zy, y_u8, **kw_)
        want = oracle.qlinear_conv(x, zx, wt, bias, mult, zy, y_u8, **kw_)
        np.testing.assert_array_equal(got, want)
        assert len(np.unique(got)) > 16  # not saturated wholesale


def test_routes_agree_at_size(env_session):
    """A ResNet-stage conv (1×256×56×56 → 256, 3×3, pad 1): GEMM and direct routes are both exact, so they
    agree bit for bit; a slab of output channels is checked against the oracle."""
    announce("qconv routes at size")
    rng = np.random.default_rng(56)
    x, zx, wt, bias, mult, *_ = make_case(rng, 1, 256, 56, 56, 256, 3, 3, 1)
    pads = (1, 1, 1, 1)
    y_gemm = run_conv(env_session(INGOT_QCONV_PATH=2), x, zx, wt, bias, mult, 17, True, pads=pads)
    y_dir = run_conv(env_session(INGOT_QCONV_PATH=1), x, zx, wt, bias, mult, 17, True, pads=pads)
    np.testing.assert_array_equal(y_gemm, y_dir)
    sl = slice(100, 108)
    want = oracle.qlinear_conv(x, zx, wt[sl], bias[sl], mult[sl], 17, True, pads=pads)
    np.testing.assert_array_equal(y_gemm[:, sl], want)
    assert len(np.unique(y_gemm)) > 64


# Depthwise strips: output widths around groups of 4, one-pixel planes, strips that split a plane and rows long
# enough to shrink them, kernel rows of one and two words, strides 1, 2 and 3, dilated kernel rows, pads wider than a
# word, a channel multiplier, 4 x 4 blocks that run over planes; then forms the strip kernel hands to the direct one (9 taps a row, dilated columns).
DEPTHWISE_CASES = [
    # n, groups, h, w, multiplier, kh, kw, strides, dilations, pads
    (2, 5, 57, 55, 1, 3, 3, (1, 1), (1, 1), (1, 1, 1, 1)),
    (3, 40, 8, 8, 1, 3, 3, (1, 1), (1, 1), (1, 1, 1, 1)),
    (2, 9, 13, 9, 2, 5, 5, (2, 2), (1, 1), (2, 2, 2, 2)),
    (1, 6, 10, 17, 1, 5, 5, (1, 1), (1, 1), (9, 11, 4, 12)),
    (1, 6, 21, 22, 1, 3, 3, (2, 2), (1, 1), (1, 9, 1, 10)),
    (1, 300, 8, 9, 1, 3, 3, (2, 2), (1, 1), (0, 0, 0, 0)),
    (1, 3, 56, 56, 1, 3, 3, (2, 2), (1, 1), (0, 0, 1, 1)),
    (1, 7, 7, 7, 1, 5, 5, (1, 1), (1, 1), (2, 2, 2, 2)),
    (1, 4, 9, 3, 2, 3, 3, (1, 1), (1, 1), (1, 1, 1, 1)),
    (1, 2, 1, 1, 3, 1, 1, (1, 1), (1, 1), (0, 0, 0, 0)),
    (1, 2, 31, 30, 1, 5, 7, (2, 2), (1, 1), (2, 3, 2, 3)),
    (1, 3, 20, 21, 1, 3, 3, (1, 3), (3, 1), (3, 1, 3, 1)),
    (1, 2, 8, 6, 1, 2, 8, (1, 1), (1, 1), (0, 6, 1, 7)),
    (1, 1, 40, 3001, 1, 3, 3, (1, 1), (1, 1), (1, 1, 1, 1)),
    (1, 1, 5, 9000, 1, 3, 3, (1, 2), (1, 1), (1, 1, 1, 1)),
    (1, 2, 12, 14, 1, 2, 9, (1, 1), (1, 1), (0, 4, 1, 4)),
    (1, 2, 12, 14, 1, 3, 3, (1, 1), (2, 2), (2, 2, 2, 2)),
]


@pytest.mark.parametrize("case", DEPTHWISE_CASES, ids=[f"d{i}" for i in range(len(DEPTHWISE_CASES))])
def test_depthwise_strips(sess, case):
    n, g, h, w, mult_c, kh, kw, st, dl, pads = case
    announce(f"qconv depthwise {case}")
    rng = np.random.default_rng(sum(case[:7]))
    for x_dtype, zx, y_u8, zy, with_bias in [(np.uint8, 131, True, 9, True), (np.uint8, 0, False, 0, False),
                                             (np.int8, -128, False, -5, True), (np.int8, 127, True, 128, False)]:
        x, zx, wt, bias, mult, *_ = make_case(rng, n, g, h, w, g * mult_c, kh, kw, g, x_dtype, zx, with_bias)
        kw_ = dict(group=g, strides=st, dilations=dl, pads=pads)
        got = run_conv(sess, x, zx, wt, bias, mult, zy, y_u8, **kw_)
        np.testing.assert_array_equal(got, oracle.qlinear_conv(x, zx, wt, bias, mult, zy, y_u8, **kw_))


@pytest.mark.parametrize("case", DEPTHWISE_CASES, ids=[f"d{i}" for i in range(len(DEPTHWISE_CASES))])
def test_depthwise_strips_forced(env_session, case):
    """The same cases where the depthwise kernels take every form they hold, however small."""
    n, g, h, w, mult_c, kh, kw, st, dl, pads = case
    announce(f"qconv depthwise forced {case}")
    rng = np.random.default_rng(sum(case[:7]) + 1)
    qs = env_session(INGOT_QCONV_PATH=4)
    for x_dtype, zx, y_u8, zy, with_bias in [(np.uint8, 131, True, 9, True), (np.int8, 127, False, -5, False)]:
        x, zx, wt, bias, mult, *_ = make_case(rng, n, g, h, w, g * mult_c, kh, kw, g, x_dtype, zx, with_bias)
        kw_ = dict(group=g, strides=st, dilations=dl, pads=pads)
        got = run_conv(qs, x, zx, wt, bias, mult, zy, y_u8, **kw_)
        np.testing.assert_array_equal(got, oracle.qlinear_conv(x, zx, wt, bias, mult, zy, y_u8, **kw_))


# Pixel GEMM: channels around whole 16-byte chunks, images narrower than a word and wider than a tile, groups whose
# channels pad, pads past the image, strides that skip columns, several images, a reduction of many k-tiles and one past
# the chunk table (which falls back to im2col).
PIXEL_CASES = [
    # n, c, h, w, m, kh, kw, g, strides, dilations, pads
    (2, 16, 9, 3, 17, 3, 3, 1, (1, 1), (1, 1), (1, 1, 1, 1)),
    (1, 15, 5, 2, 16, 3, 2, 1, (1, 1), (1, 1), (1, 0, 1, 2)),
    (3, 17, 6, 1, 33, 3, 1, 1, (2, 1), (1, 1), (1, 0, 1, 0)),
    (2, 51, 7, 130, 21, 1, 3, 3, (1, 2), (1, 1), (0, 1, 0, 1)),
    (1, 64, 8, 70, 64, 3, 3, 2, (1, 1), (2, 2), (4, 5, 2, 3)),
    (2, 33, 12, 65, 40, 1, 1, 1, (2, 2), (1, 1), (0, 0, 0, 0)),
    (1, 700, 5, 6, 24, 3, 3, 1, (1, 1), (1, 1), (1, 1, 1, 1)),
    (1, 2700, 3, 4, 16, 3, 3, 1, (1, 1), (1, 1), (1, 1, 1, 1)),
]


@pytest.mark.parametrize("path", [2, 3])
@pytest.mark.parametrize("case", PIXEL_CASES, ids=[f"p{i}" for i in range(len(PIXEL_CASES))])
def test_pixel_gemm(env_session, path, case):
    n, c, h, w, m, kh, kw, g, st, dl, pads = case
    announce(f"qconv pixel gemm {case} path={path}")
    rng = np.random.default_rng(sum(case[:7]))
    qs = env_session(INGOT_QCONV_PATH=path)
    for x_dtype, zx, y_u8, zy, with_bias in [(np.uint8, 131, True, 9, True), (np.int8, -128, False, -5, False)]:
        x, zx, wt, bias, mult, *_ = make_case(rng, n, c, h, w, m, kh, kw, g, x_dtype, zx, with_bias)
        kw_ = dict(group=g, strides=st, dilations=dl, pads=pads)
        got = run_conv(qs, x, zx, wt, bias, mult, zy, y_u8, **kw_)
        np.testing.assert_array_equal(got, oracle.qlinear_conv(x, zx, wt, bias, mult, zy, y_u8, **kw_))


# Every instance of the pixel GEMM (they differ in waves, ring depth and where the chunk table lies): pixels and channels
# off every tile's grid, groups, several images, one k-tile and more than a ring holds.
@pytest.mark.parametrize("cfg", range(7))
@pytest.mark.parametrize("case", [PIXEL_CASES[i] for i in (0, 3, 4)] +
                         [(3, 40, 11, 29, 270, 3, 3, 2, (1, 1), (1, 1), (1, 1, 1, 1)),
                          (2, 272, 5, 9, 130, 3, 3, 1, (2, 1), (1, 1), (1, 1, 1, 1))], ids=[f"t{i}" for i in range(5)])
def test_pixel_gemm_forced_tiles(env_session, cfg, case):
    n, c, h, w, m, kh, kw, g, st, dl, pads = case
    m = -(-m // g) * g
    announce(f"qconv pixel gemm tile {cfg} {case}")
    rng = np.random.default_rng(sum(case[:7]) + 2)
    qs = env_session(INGOT_QCONV_PATH=2, INGOT_GEMM_CFG=cfg)
    x, zx, wt, bias, mult, *_ = make_case(rng, n, c, h, w, m, kh, kw, g, np.uint8, 131, True)
    kw_ = dict(group=g, strides=st, dilations=dl, pads=pads)
    got = run_conv(qs, x, zx, wt, bias, mult, 9, True, **kw_)
    np.testing.assert_array_equal(got, oracle.qlinear_conv(x, zx, wt, bias, mult, 9, True, **kw_))


@pytest.mark.parametrize("path", [2, 3])
def test_images_in_two_chunks(env_session, path):
    """Images whose copies exceed the chunk's 512 MiB (three of 12.6 million pixels of 16 bytes; the column matrix of
    path 3 likewise) run in chunks that share one workspace: the oracle's bytes at both ends of every image."""
    announce(f"qconv 3 x 1 x 4096 x 3072 in chunks, path={path}")
    rng = np.random.default_rng(3072)
    x, zx, wt, bias, mult, *_ = make_case(rng, 3, 1, 4096, 3072, 16, 3, 3, 1)
    qs = env_session(INGOT_QCONV_PATH=path)
    kw_ = dict(strides=(2, 2))
    got = run_conv(qs, x, zx, wt, bias, mult, 17, True, pads=(1, 1, 1, 1), **kw_)
    assert 2 * 16 * 4096 * 3072 < 512 << 20 < 3 * 16 * 4096 * 3072 and got.shape == (3, 16, 2048, 1536)
    for i in range(3):
        top = oracle.qlinear_conv(x[i:i + 1, :, :6], zx, wt, bias, mult, 17, True, pads=(1, 1, 0, 1), **kw_)
        np.testing.assert_array_equal(got[i:i + 1, :, :3], top)
        end = oracle.qlinear_conv(x[i:i + 1, :, -7:], zx, wt, bias, mult, 17, True, pads=(0, 1, 0, 1), **kw_)
        np.testing.assert_array_equal(got[i:i + 1, :, -3:], end)


def conv_call(sess, n, c, h, w, m, ks, group, stride=1):
    """A prepared u8 convolution with pad ks // 2 on random device data: the call and a function that frees it."""
    rng = np.random.default_rng(n + c + h + m)
    oh, ow = ((d + 2 * (ks // 2) - ks) // stride + 1 for d in (h, w))
    wt = rng.integers(-128, 128, (m, c // group, ks, ks), dtype=np.int8)
    pw = sess.upload_weight(wt.reshape(m, -1), trans=True, pack_dtype=L.DT_I8)
    x = sess.to_device(rng.integers(0, 256, (n, c, h, w), dtype=np.uint8), L.DT_U8)
    mult = sess.to_device(np.full(m, 1e-3, np.float32))
    y = sess.empty(L.DT_U8, (n, m, oh, ow))

    def call():
        sess.qlinear_conv(x, 120, pw, wt.shape, mult, 128, y, group=group, strides=(stride, stride), pads=(ks // 2,) * 4)

    return call, lambda: [t.free() for t in (pw, x, mult, y)]


def conv_us(sess, *shape):
    """Least time of a pass among 40, over six runs: the host's share is the same on every route."""
    call, free = conv_call(sess, *shape)
    best = 1e30
    for _ in range(6):
        sess.timer_start()
        for _ in range(40):
            call()
        best = min(best, sess.timer_stop() * 1e3 / 40)
    free()
    return best


def assert_not_slower(env_session, shape, routes, margin):
    """The route taken by itself takes at most margin times the best of the others (at fault only if in every attempt)."""
    sessions = [env_session(INGOT_QCONV_PATH=p) for p in "0" + routes]
    for _ in range(3):
        auto, *others = (conv_us(s, *shape) for s in sessions)
        if auto < margin * min(others):
            return
    raise AssertionError(f"{auto:.1f} us, routes {routes}: {others}")


@pytest.mark.parametrize("shape", [(32, 960, 7, 7, 960, 3, 960), (64, 512, 2, 2, 512, 3, 512),
                                   (64, 512, 1, 1, 512, 1, 512), (32, 640, 7, 7, 640, 3, 640, 2),
                                   (64, 1024, 6, 6, 1024, 3, 1024), (8, 64, 56, 56, 64, 3, 64, 3)])
def test_small_depthwise_planes_not_slower_than_direct(env_session, shape):
    """Depthwise planes that give a strip's wave little to do take the direct kernel (the strip kernel needed 1.6 to 7
    times its time here)."""
    announce(f"qconv depthwise route times {shape}")
    assert_not_slower(env_session, shape, "1", 1.3)


# Shapes whose route the size rules decide: patches and strides that skip pixels of few channels, a narrow first layer,
# images of fewer pixels than the weight has rows, channel multipliers, few small depthwise planes, and ordinary layers on
# either side.
ROUTE_SHAPES = [
    # (n, c, h, w, m, ks, group, stride), the routes that hold it
    ((8, 3, 224, 224, 768, 16, 1, 16), "23"), ((8, 1, 224, 224, 32, 7, 1, 4), "23"), ((8, 3, 224, 224, 64, 7, 1, 2), "23"),
    ((1, 1024, 7, 7, 1024, 3, 1, 1), "23"), ((4, 512, 14, 14, 1024, 3, 1, 2), "23"), ((1, 256, 56, 56, 256, 3, 1, 1), "23"),
    ((1, 64, 28, 28, 1024, 3, 64, 1), "124"), ((4, 3, 64, 64, 96, 5, 3, 1), "124"), ((1, 8, 56, 56, 256, 7, 8, 1), "124"),
    ((1, 672, 7, 7, 672, 7, 672, 2), "14"), ((2, 1152, 5, 5, 1152, 7, 1152, 2), "14"), ((8, 480, 4, 4, 480, 5, 480, 1), "14"),
    ((8, 3, 64, 64, 16, 1, 1, 1), "12"), ((8, 3, 128, 128, 32, 3, 1, 1), "12"),
]


@pytest.mark.parametrize("shape,routes", ROUTE_SHAPES, ids=[f"r{i}" for i in range(len(ROUTE_SHAPES))])
def test_auto_route_not_slower(env_session, shape, routes):
    """The route taken by itself against the others that hold the shape, timed in the same run."""
    announce(f"qconv routes {shape}")
    assert_not_slower(env_session, shape, routes, 1.2)


@pytest.mark.parametrize("shape", [s for s, _ in ROUTE_SHAPES if s[1] * s[2] * s[3] * s[4] * s[5] ** 2 // s[6] < 4e8] +
                         [(2, 3, 30, 34, 40, 16, 1, 16), (1, 1, 40, 41, 32, 7, 1, 4), (1, 520, 7, 7, 530, 3, 1, 1)])
def test_routes_by_size_exact(sess, shape):
    """The same shapes (and small ones of the same kinds) by the route taken: the oracle's bytes."""
    announce(f"qconv route values {shape}")
    n, c, h, w, m, ks, group, stride = shape
    rng = np.random.default_rng(c + m)
    x, zx, wt, bias, mult, *_ = make_case(rng, min(n, 2), c, h, w, m, ks, ks, group)
    kw_ = dict(group=group, strides=(stride, stride), pads=(ks // 2,) * 4)
    got = run_conv(sess, x, zx, wt, bias, mult, 17, True, **kw_)
    np.testing.assert_array_equal(got, oracle.qlinear_conv(x, zx, wt, bias, mult, 17, True, **kw_))


def test_short_reduction_of_a_large_image(sess):
    """2^24 pixels with K below 32 (a column matrix would be refused): accepted, the oracle's bytes in the first and
    last rows."""
    announce("qconv 1 x 3 x 4096 x 4096")
    rng = np.random.default_rng(4096)
    x, zx, wt, bias, mult, *_ = make_case(rng, 1, 3, 4096, 4096, 16, 3, 3, 1)
    got = run_conv(sess, x, zx, wt, bias, mult, 17, True, pads=(1, 1, 1, 1))
    top = oracle.qlinear_conv(x[:, :, :5], zx, wt, bias, mult, 17, True, pads=(1, 1, 0, 1))
    np.testing.assert_array_equal(got[:, :, :4], top)
    end = oracle.qlinear_conv(x[:, :, -5:], zx, wt, bias, mult, 17, True, pads=(0, 1, 1, 1))
    np.testing.assert_array_equal(got[:, :, -4:], end)


def test_short_reduction_captured_on_a_fresh_session(env_session):
    """A convolution of a short reduction captured into a graph by a session without a workspace yet: it needs none
    there, and every replay gives the eager bytes."""
    import ctypes

    announce("qconv capture")
    s = env_session()
    rng = np.random.default_rng(27)
    n, c, h, w, m = 8, 3, 64, 64, 64
    x, zx, wt, bias, mult, *_ = make_case(rng, n, c, h, w, m, 3, 3, 1)
    pw = s.upload_weight(wt.reshape(m, -1), trans=True, pack_dtype=L.DT_I8)
    dx, dm, db = s.to_device(x, L.DT_U8), s.to_device(mult), s.to_device(bias)
    y = s.empty(L.DT_U8, (n, m, h, w))
    call = lambda: s.qlinear_conv(dx, zx, pw, wt.shape, dm, 17, y, bias=db, pads=(1, 1, 1, 1))
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(ln.split()[-1] for ln in f if "libamdhip64" in ln))
    st, graph, ex = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    L.check(s.lib.ingot_rocm_stream(s.h, ctypes.byref(st)))
    s.sync()
    assert s.workspace_bytes() == 0
    assert hip.hipStreamBeginCapture(st, 2) == 0  # relaxed
    call()
    assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    want = oracle.qlinear_conv(x, zx, wt, bias, mult, 17, True, pads=(1, 1, 1, 1))
    for _ in range(3):
        s.memset(y, 0)
        assert hip.hipGraphLaunch(ex, st) == 0
        np.testing.assert_array_equal(y.numpy(), want)
        s.memset(y, 0)
        call()
        np.testing.assert_array_equal(y.numpy(), want)
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)


def test_empty_and_degenerate(sess):
    announce("qconv empty")
    rng = np.random.default_rng(0)
    # no images
    x, zx, wt, bias, mult, *_ = make_case(rng, 1, 4, 5, 5, 8, 3, 3, 1)
    got = run_conv(sess, x[:0], zx, wt, bias, mult, 0, True)
    assert got.shape == (0, 8, 3, 3)
    # kernel one wider than the input: OW = (5 − 6)/1 + 1 = 0
    got = run_conv(sess, x, zx, np.ascontiguousarray(np.pad(wt, ((0, 0), (0, 0), (0, 0), (0, 3)))), bias, mult, 0,
                   True)
    assert got.shape == (1, 8, 3, 0)
    # two wider: a negative output size is an error (the reference cannot allocate it)
    with pytest.raises(IngotError, match="negative output size"):
        run_conv(sess, x, zx, np.ascontiguousarray(np.pad(wt, ((0, 0), (0, 0), (0, 0), (0, 4)))), bias, mult, 0,
                 True)
    # 1×1 image, 1×1 kernel, a single channel
    x1 = np.array([[[[200]]]], np.uint8)
    w1 = np.array([[[[-3]]]], np.int8)
    got = run_conv(sess, x1, 100, w1, None, np.array([0.5], np.float32), 7, True)
    np.testing.assert_array_equal(got, oracle.qlinear_conv(x1, 100, w1, None, np.array([0.5], np.float32), 7, True))


def test_zero_point_outside_dtype_declines(sess):
    announce("qconv decline")
    x = np.zeros((1, 1, 3, 3), np.uint8)
    w = np.ones((1, 1, 1, 1), np.int8)
    with pytest.raises(IngotError, match="outside the range"):
        run_conv(sess, x, -5, w, None, np.ones(1, np.float32), 0, True)


# ---- operator layer ----

def dev(sess, arr, code=None):
    return sess.to_device(np.ascontiguousarray(arr), code)


def op_inputs(sess, x, zx, wt, wsc, xs, ys, zy, y_dtype, bias=None):
    f32 = lambda v: dev(sess, np.asarray(v, np.float32).reshape(-1))
    ins = [dev(sess, x, DT[x.dtype]), f32([xs]), dev(sess, np.array([zx], x.dtype), DT[x.dtype]),
           dev(sess, wt, L.DT_I8), f32(wsc), dev(sess, np.zeros(wt.shape[0], np.int8), L.DT_I8), f32([ys]),
           dev(sess, np.array([zy], y_dtype), DT[np.dtype(y_dtype)])]
    if bias is not None:
        ins.append(dev(sess, bias, L.DT_I32))
    return ins


def run_op(op, *ins):
    outs = op.run(*ins)
    res = [o.numpy() for o in outs]
    for o in outs:
        o.free()
    return res


@pytest.mark.parametrize("cfg", REF_CFGS, ids=[f"c{i}" for i in range(len(REF_CFGS))])
def test_op_reference_geometries(sess, cfg):
    """TestQLinearConv through the op (ops/quant_optest_test.go:133-192): NCHW u8 in, u8 out, per-channel
    w_scale, int32 bias, attributes group/strides/pads/kernel_shape."""
    n, c, h, w, m, kh, kw, g, sh, sw, pt, pl = cfg
    announce(f"qconv op cfg {cfg}")
    rng = np.random.default_rng(7 + sum(cfg))
    x, zx, wt, bias, _, xs, wsc, ys = make_case(rng, n, c, h, w, m, kh, kw, g)
    op = sess.op("QLinearConv", 10, {"group": g, "strides": (sh, sw), "pads": (pt, pl, pt, pl),
                                     "kernel_shape": (kh, kw)})
    (y,) = run_op(op, *op_inputs(sess, x, zx, wt, wsc, xs, ys, 17, np.uint8, bias))
    mult = oracle.qconv_mult(xs, wsc, ys, m)
    want = oracle.qlinear_conv(x, zx, wt, bias, mult, 17, True, group=g, strides=(sh, sw), pads=(pt, pl, pt, pl))
    assert y.dtype == np.uint8
    np.testing.assert_array_equal(y, want)
    op.free()


@pytest.mark.parametrize("auto_pad", ["SAME_UPPER", "SAME_LOWER", "VALID"])
def test_op_auto_pad_and_s8_output(sess, auto_pad):
    announce(f"qconv op auto_pad {auto_pad}")
    rng = np.random.default_rng(99)
    x, zx, wt, _, _, xs, wsc, ys = make_case(rng, 2, 24, 11, 8, 32, 4, 3, 1, np.int8, -9, per_channel=False)
    op = sess.op("QLinearConv", 10, {"auto_pad": auto_pad, "strides": (2, 1), "dilations": (1, 2)})
    (y,) = run_op(op, *op_inputs(sess, x, zx, wt, wsc, xs, ys, -4, np.int8))
    pads = oracle.resolve_pads(auto_pad, (0, 0, 0, 0), (2, 1), (1, 2), 11, 8, 4, 3)
    want = oracle.qlinear_conv(x, zx, wt, None, oracle.qconv_mult(xs, wsc, ys, 32), -4, False, strides=(2, 1),
                               dilations=(1, 2), pads=pads)
    assert y.dtype == np.int8
    np.testing.assert_array_equal(y, want)
    op.free()


def test_op_errors(sess):
    announce("qconv op errors")
    rng = np.random.default_rng(1)
    x, zx, wt, bias, _, xs, wsc, ys = make_case(rng, 1, 4, 6, 6, 4, 3, 3, 1)
    ins = op_inputs(sess, x, zx, wt, wsc, xs, ys, 0, np.uint8, bias)
    op = sess.op("QLinearConv", 10, {"pads": (1, 1, 1, 1)})
    with pytest.raises(IngotError, match="need 8-9 inputs"):
        op.run(*ins[:5])
    with pytest.raises(IngotError, match="non-zero weight zero_point"):
        op.run(*(ins[:5] + [dev(sess, np.ones(4, np.int8), L.DT_I8)] + ins[6:]))
    with pytest.raises(IngotError, match="only s8 weights"):
        op.run(*(ins[:3] + [dev(sess, wt.view(np.uint8), L.DT_U8)] + ins[4:]))
    with pytest.raises(IngotError, match="per-tensor activation/output quantization only"):
        op.run(*(ins[:2] + [dev(sess, np.array([1, 2], np.uint8), L.DT_U8)] + ins[3:]))
    with pytest.raises(IngotError, match="only 2-D conv"):
        op.run(*([dev(sess, x.reshape(1, 4, 36), L.DT_U8)] + ins[1:]))
    op_g = sess.op("QLinearConv", 10, {"group": 3})
    with pytest.raises(IngotError, match="channel mismatch"):
        op_g.run(*ins)
    op_p = sess.op("QLinearConv", 10, {"auto_pad": "BOGUS"})
    with pytest.raises(IngotError, match="unsupported auto_pad"):
        op_p.run(*ins)
    with pytest.raises(IngotError, match="only 1-D and 2-D conv supported"):
        sess.op("QLinearConv", 10, {"strides": (1, 1, 1, 1)})
    for o in (op, op_g, op_p):
        o.free()
