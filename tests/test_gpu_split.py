"""The split-bf16 convolution tiles (fp32 products as six bf16 products): every edge of the tile against the float64
oracle with no more error than the fp32 tile of the same layer, and the inputs that a bf16 split cannot carry."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as orc  # noqa: E402

pytestmark = pytest.mark.gpu
SPLIT, FP32 = 256, 2  # OMT_TILE_SPLIT; the 64 x 128 gather tile
_CL = torch.channels_last


@pytest.fixture(scope="module")
def ops(cuda):
    from omarchy_mac_torch import hip_ops
    return hip_ops


def rnd(rng, *shape, scale=1.0):
    return (rng.standard_normal(shape) * scale).astype(np.float32)


def run(ops, d, t, x, w, gy, s, p, tile, slices=1):
    ops.set_conv_plan(d, x.shape, w.shape, s, p, tile, slices)
    y = {"fwd": lambda: ops.conv2d(t[0], t[1], None, s, p), "fwd_nhwc": lambda: ops.conv2d_nhwc(t[0], t[1], None, s, p),
         "dgrad": lambda: ops.conv2d_dgrad(t[2], t[1], x.shape, s, p),
         "dgrad_nhwc": lambda: ops.conv2d_dgrad_nhwc(t[2], t[1], x.shape, s, p)}[d]()
    return y.contiguous().cpu().numpy()


# n, ci, co, h, w, ks, stride, pad: output rows around 64 and 128 (both tile heights), pixels around 256, reductions
# with an odd half K-block (C of 16 and 48 with 9 taps), runs that cross two taps (C of 16), any channels
SHAPES = [
    (1, 16, 64, 15, 17, 3, 1, 1), (1, 48, 65, 16, 16, 3, 1, 1), (2, 32, 128, 11, 12, 1, 1, 0),
    (1, 64, 129, 257, 1, 1, 1, 0), (3, 33, 63, 9, 11, 3, 1, 1), (2, 7, 200, 10, 13, 5, 2, 2),
    (2, 80, 48, 12, 9, 3, 2, 1), (2, 128, 16, 7, 7, 3, 1, 1), (1, 3, 64, 33, 29, 7, 2, 3), (40, 17, 31, 1, 1, 1, 1, 0),
    # more tiles than CUs, so that a workgroup runs several, of one K-block and of three
    (2, 16, 64, 190, 190, 1, 1, 0), (2, 72, 40, 190, 183, 1, 1, 0),
    # window tiles (channels % 32): tiles over several images, windows of 5 and 2 rows, strided phases (grad input),
    # the super-pixel grad input, the widest rows that fit (64: 594 of 596 slots) and rows that do not
    (9, 32, 70, 7, 7, 3, 1, 1), (3, 64, 130, 14, 9, 3, 1, 1), (2, 96, 64, 20, 11, 5, 1, 2), (2, 32, 32, 9, 9, 2, 1, 0),
    (3, 32, 64, 17, 15, 3, 2, 1), (2, 3, 64, 33, 29, 11, 4, 2), (2, 32, 33, 64, 64, 3, 1, 1), (1, 32, 16, 5, 200, 3, 1, 1),
    (2, 64, 64, 5, 3, 3, 1, 3),
]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_split_tile_is_as_exact_as_the_fp32_tile(cuda, ops, shape):
    """Forward and grad input, both memory formats, 1 and 3 K slices. The float64 oracle is the reference: the split
    tile may be off by as much as the fp32 tile is, or by one rounding of the result (2^-24 each, relative)."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape))
    x, wt = rnd(rng, n, ci, h, w), rnd(rng, co, ci, ks, ks, scale=(ci * ks * ks) ** -0.5)
    y = orc.conv_fwd(x, wt, None, s, p)
    gy = rnd(rng, *y.shape)
    gx = orc.conv_dgrad(gy, wt, x.shape, s, p)
    try:
        for d, ref in (("fwd", y), ("dgrad", gx), ("fwd_nhwc", y), ("dgrad_nhwc", gx)):
            t = [torch.from_numpy(a).to(cuda) for a in (x, wt, gy)]
            t = [a.contiguous(memory_format=_CL) for a in t] if d.endswith("nhwc") else t
            for slices in (1, 3):
                e32 = orc.rel_l2(run(ops, d, t, x, wt, gy, s, p, FP32, slices), ref)
                err = orc.rel_l2(run(ops, d, t, x, wt, gy, s, p, SPLIT, slices), ref)
                assert err <= max(e32, 2.0 ** -24), (d, slices, err, e32)
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("shape", [(1, 130, 128, 5, 5, 3, 2, 1), (2, 64, 96, 7, 4, 5, 3, 2), (1, 96, 40, 3, 9, 3, 4, 1), (1, 64, 128, 7, 7, 3, 2, 0)],
                         ids=lambda s: "x".join(map(str, s)))
def test_split_k_slices_past_a_short_phase(cuda, ops, shape):
    """A strided grad input's phases sum one tap to several (or none): in as many K slices as the longest has K-blocks,
    most slices of the short ones are empty. Against the oracle; and with an infinity and a NaN in the filter, which
    reach the pixels that they reach through the fp32 tile."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape))
    x, wt = rnd(rng, n, ci, h, w), rnd(rng, co, ci, ks, ks)
    gy = rnd(rng, n, co, (h + 2 * p - ks) // s + 1, (w + 2 * p - ks) // s + 1)
    ref = orc.conv_dgrad(gy, wt, x.shape, s, p)
    try:
        for special in (False, True):
            if special:
                wt[co - 1, ci - 1, 1, 1], wt[3, 5, 0, 2] = np.inf, np.nan
            t = [torch.from_numpy(a).to(cuda) for a in (x, wt, gy)]
            tc = [a.contiguous(memory_format=_CL) for a in t]
            for d, u in (("dgrad", t), ("dgrad_nhwc", tc)):
                for slices in (3, 64):
                    a, b = (run(ops, d, u, x, wt, gy, s, p, tile, slices) for tile in (SPLIT, FP32))
                    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
                    if not special:
                        assert orc.rel_l2(a, ref) <= max(orc.rel_l2(b, ref), 2.0 ** -24), (d, slices)
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("shape", [(2, 32, 130, 9, 15, 3, 1, 1), (3, 48, 64, 10, 7, 3, 2, 1), (2, 64, 140, 8, 8, 1, 1, 0)],
                         ids=lambda s: "x".join(map(str, s)))
def test_tile_1_is_the_fp32_128x128_tile(cuda, ops, shape):
    """The split tile has its own index: tile 1 sums as the other fp32 tiles of 16-deep K-blocks do, to the bit, in every
    K order (its three variants) and channels last."""
    n, ci, co, h, w, ks, s, p = shape
    ng = ops.conv_num_tiles("fwd") // 3
    rng = np.random.default_rng(sum(shape))
    x, wt = rnd(rng, n, ci, h, w), rnd(rng, co, ci, ks, ks)
    gy = rnd(rng, n, co, (h + 2 * p - ks) // s + 1, (w + 2 * p - ks) // s + 1)
    t = [torch.from_numpy(a).to(cuda) for a in (x, wt, gy)]
    tc = [a.contiguous(memory_format=_CL) for a in t]
    try:
        for d in ("fwd", "dgrad", "fwd_nhwc", "dgrad_nhwc"):
            for v in (0, ng, 2 * ng) if d in ("fwd", "dgrad") else (0,):
                for slices in (1, 3):
                    u = tc if d.endswith("nhwc") else t
                    a, b = (run(ops, d, u, x, wt, gy, s, p, tile + v, slices) for tile in (1, 2))
                    assert np.array_equal(a, b), (d, v, slices)
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("ci", [48, 64], ids=["split", "window"])
@pytest.mark.parametrize("kind", ["inf", "nan", "huge", "tiny", "overflow"])
def test_split_tile_falls_back_on_values_it_cannot_split(cuda, ops, kind, ci):
    """Infinities, NaN, values that round past the largest bf16, sums that overflow, and inputs whose low terms
    underflow: the tile is computed again in fp32, so every output is the fp32 tile's to the bit where the whole tile
    is affected, and equal in kind (NaN, infinity, finite within rounding) elsewhere."""
    rng = np.random.default_rng(3)
    n, co, h = 2, 96, 13
    x, wt = rnd(rng, n, ci, h, h), rnd(rng, co, ci, 3, 3, scale=0.05)
    if kind in ("inf", "nan"):
        x[1, 5, 6, 7] = np.inf if kind == "inf" else np.nan
        x[0, 9, 0, 0] = -np.inf if kind == "inf" else np.nan
    elif kind == "huge":
        x[1, 5, 6, 7] = np.float32(3.4e38)
        wt *= np.float32(1e-3)
    elif kind == "overflow":
        x *= np.float32(1e30)
        wt *= np.float32(1e9)
    else:
        x *= np.float32(2.0 ** -112)
    t = [torch.from_numpy(a).to(cuda) for a in (x, wt)]
    tc = [a.contiguous(memory_format=_CL) for a in t]
    try:
        for d, u in (("fwd", t), ("fwd_nhwc", tc)):
            a = run(ops, d, u, x, wt, None, 1, 1, SPLIT)
            b = run(ops, d, u, x, wt, None, 1, 1, FP32)
            assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
            assert np.array_equal(a[np.isinf(a)], b[np.isinf(b)])
            f = np.isfinite(a)
            if kind in ("tiny", "overflow"):
                assert np.array_equal(a[f], b[f])
            else:
                scale = np.abs(b[f]).max() if kind == "huge" else np.sqrt((b[f].astype(np.float64) ** 2).mean())
                # both within K 2^-24 relative of the exact sums (K = 9 ci products)
                assert np.abs(a[f].astype(np.float64) - b[f]).max() <= 2 * 9 * ci * 2.0 ** -24 * scale
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("val", [np.inf, np.nan, 3.4e38], ids=str)
def test_one_sum_anywhere_in_a_tile_calls_for_fp32(cuda, ops, val):
    """A value that the split cannot carry in one row of the filter (or of gy), each place of a lane's four accumulator
    rows in turn: the outputs are the fp32 tile's, NaN, infinity or finite, and to the bit (one 16-deep order)."""
    rng = np.random.default_rng(5)
    n, ci, co, h = 1, 64, 64, 8
    x, wt, gy = rnd(rng, n, ci, h, h), rnd(rng, co, ci, 3, 3, scale=0.05), rnd(rng, n, co, h, h)
    try:
        for row in (0, 17, 34, 63):
            for d in ("fwd", "dgrad", "fwd_nhwc", "dgrad_nhwc", "wgrad", "wgrad_nhwc"):
                xv, wv, gv = x.copy(), wt.copy(), gy.copy()
                if d.startswith("wgrad"):
                    gv[0, row, 3, 4] = val
                elif d.startswith("dgrad"):
                    wv[5, row, 1, 1] = val
                else:
                    wv[row, 5, 1, 1] = val
                t = [torch.from_numpy(a).to(cuda) for a in (xv, wv, gv)]
                t = [a.contiguous(memory_format=_CL) for a in t] if d.endswith("nhwc") else t
                got = []
                for tile in (SPLIT, FP32):
                    if d.startswith("wgrad"):
                        ops.set_conv_plan(d, x.shape, wt.shape, 1, 1, tile, 1)
                        fn = ops.conv2d_wgrad_nhwc if d.endswith("nhwc") else ops.conv2d_wgrad
                        got.append(fn(t[0], t[2], 3, 1, 1).contiguous().cpu().numpy())
                    else:
                        got.append(run(ops, d, t, xv, wv, gv, 1, 1, tile))
                assert np.array_equal(*got, equal_nan=True), (row, d)
    finally:
        ops.clear_conv_plans()


def run_dir(ops, d, a, s, p, tile, slices=1):
    """Direction d of the layer with host arrays a = (x, w, gy) under the plan (tile, slices)."""
    t = [torch.from_numpy(np.ascontiguousarray(v)).to("cuda") for v in a]
    t = [v.contiguous(memory_format=_CL) for v in t] if d.endswith("nhwc") else t
    if not d.startswith("wgrad"):
        return run(ops, d, t, *a, s, p, tile, slices)
    ops.set_conv_plan(d, a[0].shape, a[1].shape, s, p, tile, slices)
    fn = ops.conv2d_wgrad_nhwc if d.endswith("nhwc") else ops.conv2d_wgrad
    return fn(t[0], t[2], a[1].shape[2], s, p).contiguous().cpu().numpy()


ALL_DIRS = ("fwd", "dgrad", "wgrad", "fwd_nhwc", "dgrad_nhwc", "wgrad_nhwc")
# one tile each: window, split, channel-major, strided phases, super-pixel grad input, 1x1
ONE_TILE = [(2, 64, 64, 8, 8, 3, 1, 1), (2, 48, 64, 8, 8, 3, 1, 1), (2, 33, 40, 8, 8, 3, 1, 1), (2, 48, 64, 9, 9, 3, 2, 1),
            (2, 3, 32, 33, 29, 11, 4, 2), (2, 64, 64, 8, 8, 1, 1, 0)]


@pytest.mark.parametrize("kind", ["huge_x", "huge_w", "tiny_image", "tiny_row", "subnormal"])
@pytest.mark.parametrize("shape", ONE_TILE, ids=lambda s: "x".join(map(str, s)))
def test_operands_that_lose_bits_in_the_split(cuda, ops, shape, kind):
    """Operands below 2^-109 lose bits in bf16, which shows in no sum where the other operand is huge or the rest of the
    tile is ordinary. Every direction gives the fp32 tile's outputs, to the bit (the whole tile is computed again)."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape))
    x, wt = rnd(rng, n, ci, h, w), rnd(rng, co, ci, ks, ks)
    gy = rnd(rng, n, co, (h + 2 * p - ks) // s + 1, (w + 2 * p - ks) // s + 1)
    up, down = np.float32(2.0 ** 100), np.float32(2.0 ** -119)
    try:
        for d in ALL_DIRS:
            if d == "wgrad_nhwc" and (co % 4 or ci % 8) or d == "fwd_nhwc" and ci % 16 or d == "dgrad_nhwc" and co % 16:
                continue  # not the split tile
            a = [x.copy(), wt.copy(), gy.copy()]
            # the operands: source and filter, or the two sources of the grad weight
            i, j = {"f": (0, 1), "d": (2, 1), "w": (0, 2)}[d[0]]
            if kind in ("huge_x", "huge_w"):
                i, j = (i, j) if kind == "huge_x" else (j, i)
                a[i] *= up
                a[j] *= down
            elif kind == "tiny_image":
                a[i][0] *= down
            elif kind == "tiny_row":  # of the filter's output rows; of gy
                if j == 1 and d[0] == "f":
                    a[1][5] *= down
                else:
                    a[j][:, 2] *= down
            else:
                a[i] *= np.float32(2.0 ** -110)
                a[i] *= np.float32(2.0 ** -28)
                a[j] *= np.float32(2.0 ** 110)
            slices = 2 if d[0] == "w" and kind != "tiny_image" else 1  # (an ordinary image's slice stays split)
            got = [run_dir(ops, d, a, s, p, tile, slices) for tile in (SPLIT, FP32)]
            assert np.array_equal(*got), d
            if kind != "subnormal" or d[0] == "w":
                assert np.abs(got[1]).max() > 0, d
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("shape", ONE_TILE, ids=lambda s: "x".join(map(str, s)))
def test_small_operands_that_split_exactly(cuda, ops, shape):
    """Multiples k 2^-130, |k| <= 5, are subnormal in bf16 and split exactly: against integers times 2^90 every sum is
    exact in fp32, and so is the split tile's (no test calls for the fp32 tile)."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape))
    oh, ow = (h + 2 * p - ks) // s + 1, (w + 2 * p - ks) // s + 1
    ints = [rng.integers(-5, 6, sh).astype(np.float64) for sh in ((n, ci, h, w), (co, ci, ks, ks), (n, co, oh, ow))]
    ref = [orc.conv_fwd(*(v.astype(np.float32) for v in ints[:2]), None, s, p),
           orc.conv_dgrad(ints[2].astype(np.float32), ints[1].astype(np.float32), ints[0].shape, s, p),
           orc.conv_wgrad(ints[0].astype(np.float32), ints[2].astype(np.float32), ks, s, p)]
    try:
        for d in ALL_DIRS:
            if d == "wgrad_nhwc" and (co % 4 or ci % 8) or d == "fwd_nhwc" and ci % 16 or d == "dgrad_nhwc" and co % 16:
                continue
            i, j, r = {"f": (0, 1, 0), "d": (2, 1, 1), "w": (0, 2, 2)}[d[0]]
            for lo, hi in ((i, j), (j, i)):
                a = [v.astype(np.float32) for v in ints]
                a[lo] = (ints[lo] * 2.0 ** -130).astype(np.float32)
                a[hi] = (ints[hi] * 2.0 ** 90).astype(np.float32)
                got = run_dir(ops, d, a, s, p, SPLIT)
                assert np.array_equal(got * np.float32(2.0 ** 40), np.asarray(ref[r], np.float32)), (d, lo)
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("shape", ONE_TILE[:4], ids=lambda s: "x".join(map(str, s)))
def test_products_that_underflow_beside_ordinary_ones(cuda, ops, shape):
    """One image and one filter row at 2^-70: their products are subnormal in a tile whose other sums are ordinary. Each
    output is within K 2^-24 of its sum of magnitudes, and K of the smallest float, of the exact one."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape))
    x, wt = rnd(rng, n, ci, h, w), rnd(rng, co, ci, ks, ks)
    x[0] *= np.float32(2.0 ** -70)
    wt[3] *= np.float32(2.0 ** -70)
    gy = np.zeros((n, co, (h + 2 * p - ks) // s + 1, (w + 2 * p - ks) // s + 1), np.float32)
    tx, tw = torch.from_numpy(x).double(), torch.from_numpy(wt).double()
    ref = torch.nn.functional.conv2d(tx, tw, None, s, p).numpy()
    mag = torch.nn.functional.conv2d(tx.abs(), tw.abs(), None, s, p).numpy()
    k = ci * ks * ks
    try:
        for d in ("fwd", "fwd_nhwc"):
            if d == "fwd_nhwc" and ci % 16:
                continue
            got = run_dir(ops, d, [x, wt, gy], s, p, SPLIT).astype(np.float64)
            assert (np.abs(got - ref) <= k * (2.0 ** -24 * mag + 2.0 ** -149)).all(), d
    finally:
        ops.clear_conv_plans()


def test_the_worst_operands_of_the_kept_products(cuda, ops):
    """1 + 2^-8 - 2^-17 = h + m + l with the largest m and l: the partial products left out are 2^-24 of each product,
    with one sign. Beside them at most one rounding (2^-24, relative) for each matrix instruction of a K-block (6) and
    for each K-block's addition."""
    v = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)
    try:
        for n, ci, co, h, ks, p in ((1, 64, 64, 16, 3, 1), (1, 48, 64, 16, 1, 0), (1, 128, 130, 16, 1, 0)):
            a = [np.full((n, ci, h, h), v), np.full((co, ci, ks, ks), v), np.full((n, co, h, h), v)]
            taps = np.ones((1, 1, ks, ks), np.float32)
            count = orc.conv_fwd(np.ones((n, 1, h, h), np.float32), taps, None, 1, p).astype(np.float64)  # taps inside
            for d, ref, k in (("fwd", count * ci, ci * ks * ks), ("dgrad", count * co, co * ks * ks),
                              ("wgrad", None, h * h)):
                got = run_dir(ops, d, a, 1, p, SPLIT).astype(np.float64)
                if d == "wgrad":
                    side = np.array([h - abs(i - ks // 2) for i in range(ks)], np.float64)
                    ref = np.outer(side, side)
                exact = ref * float(v) ** 2
                assert (np.abs(got - exact) <= (1 + 6 + -(-k // 32)) * 2.0 ** -24 * exact).all(), d
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("shape", [(2, 32, 31, 9, 9, 3, 1, 1), (2, 24, 64, 9, 8, 3, 2, 1), (2, 1030, 70, 5, 7, 1, 1, 0),
                                   (2, 232, 72, 6, 6, 3, 1, 1), (1, 40, 130, 9, 9, 1, 1, 0), (3, 16, 256, 80, 80, 1, 1, 0)],
                         ids=lambda s: "x".join(map(str, s)))
def test_bn_loader_beside_a_split_plan(cuda, ops, shape):
    """Each fp32 tile that the BN loader runs where the plan is the split tile (by rows, reduction and grid), with bias
    and ReLU, against the oracle: both within K 2^-24 of the sum of magnitudes and the rounding of the loader."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape))
    x, wt, b = rnd(rng, n, ci, h, w), rnd(rng, co, ci, ks, ks, scale=(ci * ks * ks) ** -0.5), rnd(rng, co)
    bn = [rnd(rng, ci, scale=0.2), np.abs(rnd(rng, ci)) + np.float32(0.5), rnd(rng, ci), rnd(rng, ci)]
    c = [v.reshape(1, -1, 1, 1).astype(np.float64) for v in bn]
    z = np.maximum((x - c[0]) / np.sqrt(c[1] + 1e-5) * c[2] + c[3], 0).astype(np.float32)
    ref = np.maximum(orc.conv_fwd(z, wt, b, s, p), 0)
    dev = [torch.from_numpy(v).to(cuda) for v in (x, wt, b, *bn)]
    try:
        ops.set_conv_plan("fwd", x.shape, wt.shape, s, p, SPLIT, 1)
        y = ops.conv2d(dev[0], dev[1], dev[2], s, p, relu=True, bn=dev[3:]).cpu().numpy()
        assert orc.rel_l2(y, ref) <= 1e-5  # up to 2310 products' roundings and five of the loader's, random signs
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("shape", [(2, 64, 64, 8, 8, 3, 1, 1), (2, 48, 64, 8, 8, 3, 1, 1), (2, 64, 64, 9, 9, 3, 2, 1)],
                         ids=lambda s: "x".join(map(str, s)))
def test_a_redone_tile_goes_through_every_epilogue(cuda, ops, shape):
    """Tiles computed again in fp32 (tiny filter, huge source): three K slices' partials, bias and ReLU, and epilogue
    statistics are the fp32 tile's, to the bit."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape))
    x, wt, b = rnd(rng, n, ci, h, w) * np.float32(2.0 ** 100), rnd(rng, co, ci, ks, ks) * np.float32(2.0 ** -110), rnd(rng, co)
    gy = rnd(rng, n, co, (h + 2 * p - ks) // s + 1, (w + 2 * p - ks) // s + 1) * np.float32(2.0 ** 100)
    t = [torch.from_numpy(v).to(cuda) for v in (x, wt, b)]
    tc = [v.contiguous(memory_format=_CL) for v in t[:2]] + t[2:]
    try:
        if ci == 64:  # both tiles' slices end at the same K
            for d in ("fwd", "dgrad", "fwd_nhwc", "dgrad_nhwc"):
                got = [run_dir(ops, d, [x, wt, gy], s, p, tile, 3) for tile in (SPLIT, FP32)]
                assert np.array_equal(*got), d
        got = []
        for tile in (SPLIT, FP32):
            for d in ("fwd", "fwd_nhwc"):
                ops.set_conv_plan(d, x.shape, wt.shape, s, p, tile, 1)
            y, st, groups = ops.conv2d_stats(t[0], t[1], s, p)
            got.append([ops.conv2d(*t, s, p, relu=True), ops.conv2d_nhwc(*tc, s, p, relu=True), y, st[:, :groups]])
        for u, v in zip(*got):
            assert torch.equal(u, v) and float(u.abs().max()) > 0
    finally:
        ops.clear_conv_plans()


def test_a_workgroup_redoes_all_its_tiles(cuda, ops):
    """283 tiles on 256 CUs: a NaN in one of them has its workgroup compute all its tiles again in fp32."""
    rng = np.random.default_rng(11)
    x, wt = rnd(rng, 2, 16, 190, 190), rnd(rng, 64, 16, 1, 1)
    x[0, 3, 1, 2], x[1, 7, 189, 189] = np.nan, np.inf
    t = [torch.from_numpy(a).to(cuda) for a in (x, wt)]
    try:
        a = run(ops, "fwd", t, x, wt, None, 1, 0, SPLIT)
        b = run(ops, "fwd", t, x, wt, None, 1, 0, FP32)
    finally:
        ops.clear_conv_plans()
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
    f = np.isfinite(b)  # both within K 2^-24 relative of the exact sums of up to K = 16 products of a few units each
    assert np.abs(a[f].astype(np.float64) - b[f]).max() <= 2 * 16 * 2.0 ** -24 * np.abs(b[f]).max()


WFP32 = 2  # grad-weight tile
# rows around 64, 128 and 256, columns around 64, 128 and 256 (all five tile shapes); reductions that end inside a
# K-block; the orders by channels: % 32 (columns by 32 channels), % 8 (tap-major), others (element by element); 1x1
# planes of a multiple of 4 that is none of 8 (runs of four pixels that change image)
WSHAPES = [
    (3, 32, 64, 9, 11, 3, 1, 1), (2, 64, 128, 8, 8, 3, 1, 1), (2, 40, 130, 9, 9, 3, 2, 1), (1, 13, 65, 12, 10, 3, 1, 1),
    (3, 130, 256, 6, 6, 1, 1, 0), (5, 64, 300, 2, 6, 1, 1, 0), (2, 72, 260, 7, 7, 1, 1, 0), (1, 3, 48, 30, 31, 7, 2, 3),
    (2, 256, 64, 5, 5, 1, 1, 0), (1, 8, 16, 3, 3, 3, 1, 1),
]


# a last unit of gy rows that is not whole: P % 8 != 0 (channels last P % 8 == 4), few rows and one past a tile's edge,
# one image, in each column order
ROW_EDGES = [
    (1, 32, 1, 12, 11, 3, 1, 1), (1, 24, 3, 12, 11, 3, 1, 1), (1, 12, 5, 9, 13, 3, 2, 1), (1, 64, 3, 8, 9, 1, 1, 0),
    (1, 40, 4, 9, 9, 3, 1, 1), (1, 32, 12, 12, 11, 3, 1, 1), (1, 32, 129, 7, 7, 3, 1, 1), (1, 32, 132, 7, 7, 3, 1, 1),
    (1, 300, 68, 7, 7, 1, 1, 0),
]


@pytest.mark.parametrize("shape", ROW_EDGES, ids=lambda s: "x".join(map(str, s)))
def test_split_grad_weight_reads_no_row_past_the_last(cuda, ops, shape):
    """gy lies in front of NaNs in one allocation: a row past gy's last, though not stored, would have the tile computed
    again in fp32, whose sums differ. The result is that of gy alone, to the bit, and as exact as the fp32 tile's."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape) + 3)
    x, wt = rnd(rng, n, ci, h, w), rnd(rng, co, ci, ks, ks)
    gy = rnd(rng, *orc.conv_fwd(x, wt, None, s, p).shape)
    ref = orc.conv_wgrad(x, gy, ks, s, p)
    try:
        for d, fn in (("wgrad", ops.conv2d_wgrad), ("wgrad_nhwc", ops.conv2d_wgrad_nhwc)):
            nhwc = d == "wgrad_nhwc"
            if nhwc and (co % 4 or ci % 8):
                continue
            tx, tg = (torch.from_numpy(a).to(cuda).contiguous(memory_format=_CL if nhwc else torch.contiguous_format)
                      for a in (x, gy))
            buf = torch.full((gy.size + 8 * gy[0, 0].size + 64,), float("nan"), device=cuda)
            view = buf[:gy.size].view(n, *gy.shape[2:], co).permute(0, 3, 1, 2) if nhwc else buf[:gy.size].view(gy.shape)
            view.copy_(tg)
            got = []
            for tile, g in ((SPLIT, tg), (SPLIT, view), (WFP32, tg)):
                ops.set_conv_plan(d, x.shape, wt.shape, s, p, tile, 1)
                got.append(fn(tx, g, ks, s, p).contiguous().cpu().numpy())
            assert np.array_equal(got[0], got[1]), d
            err, e32 = orc.rel_l2(got[0], ref), orc.rel_l2(got[2], ref)
            assert err <= max(e32, 2.0 ** -24), (d, err, e32)
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("shape", WSHAPES, ids=lambda s: "x".join(map(str, s)))
def test_split_grad_weight_is_as_exact_as_the_fp32_tile(cuda, ops, shape):
    """Both memory formats, 1 and 3 K slices, against the float64 oracle: off by no more than the fp32 tile, or one
    rounding of the result."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape) + 1)
    x, wt = rnd(rng, n, ci, h, w), rnd(rng, co, ci, ks, ks)
    gy = rnd(rng, *orc.conv_fwd(x, wt, None, s, p).shape)
    ref = orc.conv_wgrad(x, gy, ks, s, p)
    try:
        for d, fn in (("wgrad", ops.conv2d_wgrad), ("wgrad_nhwc", ops.conv2d_wgrad_nhwc)):
            if d == "wgrad_nhwc" and co % 4:
                continue  # not covered channels-last
            t = [torch.from_numpy(a).to(cuda) for a in (x, gy)]
            t = [a.contiguous(memory_format=_CL) for a in t] if d == "wgrad_nhwc" else t
            for slices in (1, 3):
                ops.set_conv_plan(d, x.shape, wt.shape, s, p, WFP32, slices)
                e32 = orc.rel_l2(fn(t[0], t[1], ks, s, p).contiguous().cpu().numpy(), ref)
                ops.set_conv_plan(d, x.shape, wt.shape, s, p, SPLIT, slices)
                err = orc.rel_l2(fn(t[0], t[1], ks, s, p).contiguous().cpu().numpy(), ref)
                assert err <= max(e32, 2.0 ** -24), (d, slices, err, e32)
    finally:
        ops.clear_conv_plans()


@pytest.mark.parametrize("shape", [(2, 32, 70, 9, 9, 3, 1, 1), (2, 24, 70, 9, 9, 3, 1, 1), (2, 12, 64, 9, 9, 3, 1, 1),
                                   (2, 70, 68, 8, 8, 1, 1, 0)], ids=lambda s: "x".join(map(str, s)))
def test_split_grad_weight_falls_back_on_values_it_cannot_split(cuda, ops, shape):
    """Every column order of the tile: an infinity and a NaN reach the same weights as through the fp32 tile, and
    inputs whose low terms underflow give the fp32 tile's sums to the bit (both sum each K slice in the same order)."""
    n, ci, co, h, w, ks, s, p = shape
    rng = np.random.default_rng(sum(shape) + 2)
    x, gy = rnd(rng, n, ci, h, w), rnd(rng, n, co, h + 2 * p - ks + 1, w + 2 * p - ks + 1)
    try:
        for kind in ("special", "tiny"):
            a = x * np.float32(2.0 ** -112) if kind == "tiny" else x.copy()
            if kind == "special":
                a[0, 3, 4, 4], a[1, 5, 2, 2] = np.inf, np.nan
            for d, fn in (("wgrad", ops.conv2d_wgrad), ("wgrad_nhwc", ops.conv2d_wgrad_nhwc)):
                if d == "wgrad_nhwc" and co % 4:
                    continue
                t = [torch.from_numpy(v).to(cuda) for v in (a, gy)]
                t = [v.contiguous(memory_format=_CL) for v in t] if d == "wgrad_nhwc" else t
                got = []
                for tl in (SPLIT, WFP32):
                    ops.set_conv_plan(d, x.shape, (co, ci, ks, ks), s, p, tl, 2)
                    got.append(fn(t[0], t[1], ks, s, p).contiguous().cpu().numpy())
                assert np.array_equal(np.isnan(got[0]), np.isnan(got[1]))
                assert np.array_equal(np.isinf(got[0]), np.isinf(got[1]))
                f = np.isfinite(got[1])
                if kind == "tiny":
                    assert np.array_equal(got[0], got[1])
                else:  # both within K 2^-24 relative of the exact sums (K = 162 products)
                    scale = np.sqrt((got[1][f].astype(np.float64) ** 2).mean())
                    assert np.abs(got[0][f].astype(np.float64) - got[1][f]).max() <= 2 * 162 * 2.0 ** -24 * scale
    finally:
        ops.clear_conv_plans()
