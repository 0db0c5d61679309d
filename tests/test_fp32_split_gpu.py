"""The FP32 form's convs (every value as three BF16 parts on BF16 MFMA)
against the FP64 oracle, over the shapes and batch sizes where the kernel
changes: channel counts around its blocks of 16 and chunks of 32, 5x5 and
3x3 filters first and later, batches that take pieces of ten rows, five rows
and few channels, byte planes that are not 0 / 1, weights of any scale.

Bar: the parts hold FP32 values exactly and drop 2^-24 of a product at most
(see test_dropped_partial_products), and the sums of very small products are
formed again in FP32, so a conv errs like an FP32 one: K^(1/2) roundings of
2^-24 on sums of K <= 5 * 5 * 160 terms, 4e-6 a layer at worst, six layers at
most here: 2e-5 of the largest logit.
"""
import numpy as np
import pytest

# (filter, cin, cout) of the trunk and head.
NETS = {
    "narrow": [(3, 5, 7), (5, 7, 17), (3, 17, 1)],
    "odd": [(5, 22, 33), (3, 33, 48), (5, 48, 40), (3, 40, 1)],
    "wide": [(3, 40, 160), (3, 160, 130), (3, 130, 96), (3, 96, 1)],
    "reference_head": [(5, 32, 96), (3, 96, 128), (3, 128, 64), (3, 64, 1)],
}


def _table(name, scale):
    rng = np.random.default_rng(len(name))
    shapes = NETS[name]
    table = []
    for i, (f, cin, cout) in enumerate(shapes):
        std = np.sqrt(2.0 / (cin * f * f))
        # The first conv's weights carry `scale`, the last one's its inverse.
        std *= scale if i == 0 else 1 / scale if i == len(shapes) - 1 else 1
        w = rng.normal(0, std, (cout, cin, f, f)).astype(np.float32)
        b = rng.normal(0, 0.1 * (scale if i < len(shapes) - 1 else 1),
                       cout).astype(np.float32)
        # ReLU keeps the scale from layer to layer.
        act = 1 if cout > 1 else 2
        table.append({"kind": "conv", "filter": f, "cin": cin, "cout": cout,
                      "w": w, "b": b, "act": act, "bn": None})
    return table


def _bf16(x):
    """Rounded to BF16, to nearest even (finite values)."""
    u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000
    return u.astype(np.uint32).view(np.float32)


def _parts(x):
    h = _bf16(x)
    m = _bf16(x - h)
    return h, m, _bf16(x - h - m)


def test_dropped_partial_products():
    """On the CPU: three parts add up to the value exactly from 2^-103 up,
    each a BF16 normal number or 0, and six of the nine partial products to
    the product within 2^-24 of it."""
    rng = np.random.default_rng(0)
    x, y = (rng.standard_normal(1 << 20).astype(np.float32) for _ in range(2))
    x = np.concatenate([x, rng.uniform(1, 2, 1 << 20).astype(np.float32)])
    y = np.concatenate([y, rng.uniform(1, 2, 1 << 20).astype(np.float32)])
    for v in (x, np.abs(x) * np.float32(2.0 ** -102) + np.float32(2.0 ** -103)):
        p = _parts(v)
        assert (sum(q.astype(np.float64) for q in p) == v).all()
        assert all(((q == 0) | (np.abs(q) >= 2.0 ** -126)).all() for q in p)
    a, b = _parts(x), _parts(y)
    got = sum(a[i].astype(np.float64) * b[j]
              for i, j in ((0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)))
    want = x.astype(np.float64) * y
    assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("name,n,scale", [
    ("narrow", 1, 1.0), ("narrow", 67, 1.0), ("odd", 1, 1.0),
    ("odd", 33, 1.0), ("odd", 300, 1.0), ("wide", 2, 1.0), ("wide", 64, 1.0),
    ("wide", 130, 1.0), ("reference_head", 96, 1.0),
    ("reference_head", 257, 1.0), ("odd", 3, 1e30), ("odd", 3, 1e-25),
    ("odd", 3, 1e-33), ("reference_head", 130, 1e-35), ("odd", 3, 1e-37),
    ("reference_head", 3, 1e-37)])
def test_fp32_form_matches_fp64(name, n, scale):
    import leela_amd
    import oracle
    from leela_amd import caffe_weights as cw
    from leela_amd import nets
    print(f"case: {name} n={n} scale={scale}", flush=True)
    table = _table(name, scale)
    rng = np.random.default_rng(n)
    planes = (rng.random((n, table[0]["cin"], 361)) < 0.3).astype(np.uint8)
    planes[0] *= rng.integers(0, 256, planes[0].shape, dtype=np.uint8)
    be = leela_amd.Backend(0)
    try:
        cw.push_layers(be, leela_amd.NET_POLICY, table)
        be.load_net(leela_amd.NET_VALUE, nets.weight_set("A")[1])
        be.finalize()
        be.set_temperature(1.0)
        raw, _ = be.forward(leela_amd.NET_POLICY, leela_amd.PREC_FP32, planes)
    finally:
        be.close()
    oracle.load_blas()
    want, _ = oracle.forward_f64(oracle.Net.from_table(table), planes,
                                 oracle.HEAD_POLICY, temperature=1.0,
                                 gemm=True)
    for got, ref in zip(raw, want):  # (board 0 has inputs up to 255)
        assert np.abs(got - ref).max() < 2e-5 * np.abs(ref).max()


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,n", [(2, 1), (3, 5), (64, 2), (256, 4),
                                      (258, 9), (300, 3), (513, 1)])
def test_value_head_matches_fp64(hidden, n):
    """The inner-product head at hidden sizes that are and are not multiples
    of four or of the 256 units a pass holds, and batches that fill its
    four-board workgroups or not. Sums of 361 and `hidden` products: FP32
    roundings of 2^-24 * sqrt(361 * hidden) at most, 3e-5 of the result's
    scale. (Not one unit: the oracle's first product then has no ELU, as the
    reference's has none with one output.)"""
    import leela_amd
    import oracle
    from leela_amd import nets
    print(f"case: hidden={hidden} n={n}", flush=True)
    rng = np.random.default_rng(hidden)

    def layer(kind, f, cin, cout):
        k = cin * max(f, 1) ** 2
        w = rng.normal(0, np.sqrt(2.0 / k), cout * k).astype(np.float32)
        w = w.reshape((cout, cin, f, f) if kind == nets.CONV else (cout, cin))
        return (kind, f, cin, cout, w,
                rng.normal(0, 0.1, cout).astype(np.float32))

    val = [layer(nets.CONV, 3, 32, 16), layer(nets.CONV, 3, 16, 1),
           layer(nets.FC, 0, 361, hidden), layer(nets.FC, 0, hidden, 1)]
    planes = (rng.random((n, 32, 361)) < 0.3).astype(np.uint8)
    be = leela_amd.Backend(0)
    try:
        be.load_net(leela_amd.NET_POLICY, nets.weight_set("A")[0])
        be.load_net(leela_amd.NET_VALUE, val)
        be.finalize()
        raw, out = be.forward(leela_amd.NET_VALUE, leela_amd.PREC_FP32, planes)
    finally:
        be.close()
    oracle.load_blas()
    raw64, out64 = oracle.forward_f64(oracle.Net(val), planes,
                                      oracle.HEAD_VALUE, gemm=True)
    bar = 3e-5 * max(1.0, np.abs(raw64).max())
    assert np.abs(raw.ravel() - raw64.ravel()).max() < bar
    assert np.abs(out.ravel() - out64.ravel()).max() < bar


def _conv_f32(x, w, b):
    """Same-padded conv in FP32, term by term, as a matrix product with zero
    columns off the board forms it: x [n][cin][19][19]."""
    n, cin = x.shape[:2]
    cout, _, f, _ = w.shape
    h = f // 2
    xp = np.zeros((n, cin, 19 + 2 * h, 19 + 2 * h), np.float32)
    xp[:, :, h:h + 19, h:h + 19] = x
    out = np.zeros((n, cout, 19, 19), np.float32)
    for c in range(cin):
        for dy in range(f):
            for dx in range(f):
                out += (w[:, c, dy, dx][None, :, None, None] *
                        xp[:, c, dy:dy + 19, dx:dx + 19][:, None])
    return out + b[None, :, None, None]


def _same(got, want, what):
    """Infinities and NaNs where FP32 has them, the rest as above."""
    for name, f in (("nan", np.isnan), ("+inf", lambda v: v == np.inf),
                    ("-inf", lambda v: v == -np.inf)):
        np.testing.assert_array_equal(f(got), f(want), err_msg=what + name)
    ok = np.isfinite(want)
    if ok.any():
        assert np.abs(got[ok] - want[ok]).max() <= (
            2e-5 * np.abs(want[ok]).max()), what


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 130])
@pytest.mark.parametrize("kind", ["activation", "overflow", "weight",
                                  "head_weight", "nan_weight"])
@pytest.mark.parametrize("act", [1, 2])
def test_infinities_are_those_of_float32(n, kind, act):
    """Sums that overflow, infinite and NaN activations and weights, with ReLU
    (which turns a NaN into 0) and with no activation of the trunk: every logit
    is infinite, NaN or finite as in FP32, and the finite ones agree. One point
    of every board overflows (or one weight does not hold a number), so most
    of a board stays finite. n = 1 and 130: pieces of five and ten rows."""
    import leela_amd
    from leela_amd import caffe_weights as cw
    from leela_amd import nets
    print(f"case: {kind} n={n} act={act}", flush=True)
    rng = np.random.default_rng(5)
    shapes = [(5, 3, 40), (3, 40, 33), (3, 33, 1)]
    table = []
    for f, cin, cout in shapes:
        w = rng.normal(0, np.sqrt(2 / (cin * f * f)), (cout, cin, f, f))
        table.append({"kind": "conv", "filter": f, "cin": cin, "cout": cout,
                      "w": w.astype(np.float32), "bn": None,
                      "act": act if cout > 1 else 2,
                      "b": rng.normal(0, 0.1, cout).astype(np.float32)})
    planes = np.zeros((n, 3, 361), np.uint8)
    planes[:, 0] = rng.random((n, 361)) < 0.3
    w0, w1, w2 = (t["w"] for t in table)
    # Channel 7 answers to plane 2, set at one point, at that point only.
    w0[:, 2] = 0
    w0[7] = 0
    np.abs(w2, out=w2)
    planes[:, 2, 23] = 255
    if kind == "activation":
        w0[7, 2, 2, 2] = 3e38
        w1[4, 7] = 0  # 0 x inf
    elif kind == "overflow":
        # Finite activations whose products are far past FP32's range.
        w0[7, 2, 2, 2] = 1e36
        w1[:, 7] *= 1e12
    elif kind == "weight":
        w1[3, 7, 0, 2] = np.inf
        w1[5, 6, 1, 1] = -np.inf
    elif kind == "head_weight":
        w2[0, 3, 2, 0] = np.inf
    else:
        w1[9, 2, 1, 0] = np.nan
    be = leela_amd.Backend(0)
    try:
        cw.push_layers(be, leela_amd.NET_POLICY, table)
        be.load_net(leela_amd.NET_VALUE, nets.weight_set("A")[1])
        be.finalize()
        be.set_temperature(1.0)
        raw, _ = be.forward(leela_amd.NET_POLICY, leela_amd.PREC_FP32, planes)
    finally:
        be.close()
    x = planes.reshape(n, 3, 19, 19).astype(np.float32)
    with np.errstate(all="ignore"):
        for t in table:
            x = _conv_f32(x, t["w"], t["b"])
            if t["act"] == 1:
                x = np.where(x > 0, x, np.float32(0))
    want = x.reshape(n, 361)
    if kind != "nan_weight" or act == 2:
        assert not np.isfinite(want).all()
    _same(raw, want, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("hidden", [64, 258])
def test_infinite_value_head_weights(hidden):
    """An infinite weight of the last input of the first inner product makes
    its unit infinite, and the value 0, 1 or NaN as in FP32."""
    import leela_amd
    from leela_amd import nets
    print(f"case: hidden={hidden}", flush=True)
    rng = np.random.default_rng(2)
    w1 = np.abs(rng.normal(0, 0.1, (hidden, 361))).astype(np.float32)
    w1[5, 360] = np.inf
    w2 = rng.normal(0, 0.1, (1, hidden)).astype(np.float32)
    head = rng.normal(0, 0.1, (1, 4, 3, 3)).astype(np.float32)
    val = [(nets.CONV, 3, 32, 4, rng.normal(0, 0.1, (4, 32, 3, 3)).astype(
                np.float32), np.zeros(4, np.float32)),
           (nets.CONV, 3, 4, 1, head, np.full(1, 0.5, np.float32)),
           (nets.FC, 0, 361, hidden, w1, np.zeros(hidden, np.float32)),
           (nets.FC, 0, hidden, 1, w2, np.zeros(1, np.float32))]
    planes = np.zeros((5, 32, 361), np.uint8)
    be = leela_amd.Backend(0)
    try:
        be.load_net(leela_amd.NET_POLICY, nets.weight_set("A")[0])
        be.load_net(leela_amd.NET_VALUE, val)
        be.finalize()
        raw, _ = be.forward(leela_amd.NET_VALUE, leela_amd.PREC_FP32, planes)
    finally:
        be.close()
    # Empty planes: h0 is 0.5 everywhere, unit 5 +inf.
    want = np.inf if w2[0, 5] > 0 else -np.inf
    np.testing.assert_array_equal(raw.ravel(), np.full(5, want, np.float32))
