"""The layered form of the 16-bit kernels (fused_forward_layered: one launch
per conv, each conv of a board split over workgroups of output channels)
against the persistent fused kernel: the same outputs bit for bit for both
nets, both 16-bit forms and batch sizes 1..64, directly and through the
leaf queue's smallest bucket; and its latency for small batches."""
import time

import numpy as np
import pytest

from leela_amd.positions import make_batch

pytestmark = pytest.mark.gpu


def _backend(weights):
    import leela_amd
    b = leela_amd.Backend(0)
    pol, val = weights
    b.load_net(leela_amd.NET_POLICY, pol)
    b.load_net(leela_amd.NET_VALUE, val)
    b.finalize()
    return b


@pytest.fixture(scope="module")
def be(weights_a):
    b = _backend(weights_a)
    yield b
    b.close()


@pytest.fixture(scope="module")
def be_default(weights_a):
    """A backend whose layered limit is never set."""
    b = _backend(weights_a)
    yield b
    b.close()


@pytest.mark.parametrize("prec", ["bf16", "fp16"])
@pytest.mark.parametrize("n", [1, 7, 64])
def test_layered_equals_fused(be, prec, n):
    import leela_amd
    p = leela_amd.PRECISIONS[prec]
    print(f"case: {prec} n={n}", flush=True)
    for net, seed in ((leela_amd.NET_POLICY, 11), (leela_amd.NET_VALUE, 12)):
        planes = make_batch(n, seed0=seed * 1000 + n, net=net)
        be.set_layered_max(64)
        raw_l, out_l = be.forward(net, p, planes)
        be.set_layered_max(0)
        raw_f, out_f = be.forward(net, p, planes)
        be.set_layered_max(64)
        np.testing.assert_array_equal(raw_l, raw_f)
        np.testing.assert_array_equal(out_l, out_f)


@pytest.mark.parametrize("n", [2, 16, 17, 25, 26])
def test_layered_equals_fused_where_bands_split(be, n):
    """Small batches run a band's channels in two workgroups (policy up to 25
    boards, value up to 16): the same bits as the persistent kernels."""
    import leela_amd
    print(f"case: n={n}", flush=True)
    for prec in (leela_amd.PREC_BF16, leela_amd.PREC_FP16):
        for net in (leela_amd.NET_POLICY, leela_amd.NET_VALUE):
            planes = make_batch(n, seed0=7000 + n, net=net)
            be.set_layered_max(64)
            got = be.forward(net, prec, planes)
            be.set_layered_max(0)
            want = be.forward(net, prec, planes)
            be.set_layered_max(64)
            for a, b in zip(got, want):
                np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n", [65, 96, 97, 256, 257, 352, 353, 513, 600])
def test_rest_of_a_policy_batch_equals_fused(be, be_default, n):
    """Policy batches of up to 96 boards, and up to 96 boards past whole
    passes of 256, run in the layered form: the same bits as the persistent
    kernel's alone, in every row and not past them; also without a raw
    output."""
    import torch
    import leela_amd
    p = leela_amd.PREC_BF16
    print(f"case: n={n}", flush=True)
    planes = torch.from_numpy(make_batch(n, seed0=5000 + n)).cuda()
    got = {}
    be.set_layered_max(0)
    for lm, b in ((0, be), (64, be_default)):
        raw = torch.full((n + 1, 361), -7.0, device="cuda")
        out = torch.full((n + 1, 361), -7.0, device="cuda")
        only = torch.full((n + 1, 361), -7.0, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        b.forward_device(0, p, n, planes.data_ptr(), raw.data_ptr(),
                         out.data_ptr(), st)
        b.forward_device(0, p, n, planes.data_ptr(), None, only.data_ptr(),
                         st)
        got[lm] = [t.cpu().numpy() for t in (raw, out, only)]
    be.set_layered_max(64)
    for a, b in zip(got[0], got[64]):
        np.testing.assert_array_equal(a, b)
        assert (b[n] == -7.0).all()


@pytest.mark.parametrize("n,limit", [(80, 64), (272, 16), (272, 64)])
def test_a_limit_that_is_set_holds(be, be_default, n, limit):
    """Policy batches past a limit that the caller has set run in the
    persistent kernel as a whole, as they do with the limit 0; the default
    takes the 80 boards, or the 16 past a pass, in the layered form (0.8 of
    the time)."""
    import torch
    import leela_amd
    print(f"case: n={n} limit={limit}", flush=True)
    planes = torch.from_numpy(make_batch(n, seed0=3)).cuda()
    raw = torch.empty((n, 361), device="cuda")
    out = torch.empty_like(raw)
    st = torch.cuda.current_stream().cuda_stream

    def ms(b):
        return min(float(np.sum(b.forward_timed(
            0, leela_amd.PREC_FP16, n, planes.data_ptr(), raw.data_ptr(),
            out.data_ptr(), st))) for _ in range(20))

    be.set_layered_max(0)
    ms(be)  # (clocks up)
    persistent = ms(be)
    be.set_layered_max(limit)
    limited = ms(be)
    be.set_layered_max(64)
    default = ms(be_default)
    print(f"ms: {persistent:.4f} {limited:.4f} {default:.4f}", flush=True)
    assert default < 0.95 * persistent
    assert limited > (persistent + default) / 2


def test_layered_queue_bucket_equals_direct(be):
    """16 positions through the queue's 64-board bucket (layered graph,
    device-side count) equal a direct fused forward of the same boards."""
    import leela_amd
    p = leela_amd.PREC_FP16
    planes = make_batch(16, seed0=777)
    be.set_layered_max(0)
    want_raw, want = be.forward(leela_amd.NET_POLICY, p, planes)
    be.set_layered_max(64)
    from leela_amd.backend import DONE_FN
    got = np.full((16, 361), np.nan, np.float32)
    status = np.full(16, -99, np.int32)

    def done(user, st, raw, out):
        i = int(user or 0)
        status[i] = st
        if st == 0:
            got[i] = np.ctypeslib.as_array(out, (361,))
    cb = DONE_FN(done)
    be.queue_start(p, 64, 2000)
    try:
        for rep in range(3):  # graph replays with eager work between
            got[:] = np.nan
            for i in range(16):
                be.submit(leela_amd.NET_POLICY, planes[i], cb, i)
            be.join()
            assert (status == 0).all()
            np.testing.assert_array_equal(got, want)
            be.forward(leela_amd.NET_VALUE, p, make_batch(3, seed0=rep + 1,
                                                         net=1))
    finally:
        be.queue_stop()


def test_layered_latency(be):
    """Small-batch latency of the two forms (printed; the layered form must
    not be slower at one board)."""
    import torch
    import leela_amd
    dev = torch.device("cuda", 0)
    p = leela_amd.PREC_FP16
    res = {}
    for n in (1, 16, 64):
        planes = torch.from_numpy(make_batch(n, seed0=5)).to(dev)
        raw = torch.empty((n, 361), device=dev)
        out = torch.empty_like(raw)
        st = torch.cuda.current_stream(dev).cuda_stream
        for lm in (0, 64):
            be.set_layered_max(lm)
            for _ in range(3):
                be.forward_device(0, p, n, planes.data_ptr(), raw.data_ptr(),
                                  out.data_ptr(), st)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            reps = 20
            for _ in range(reps):
                be.forward_device(0, p, n, planes.data_ptr(), raw.data_ptr(),
                                  out.data_ptr(), st)
            torch.cuda.synchronize()
            res[(n, lm)] = (time.perf_counter() - t0) / reps * 1e6
    be.set_layered_max(64)
    print("policy fp16 latency (us): " + ", ".join(
        f"n={n} fused {res[(n, 0)]:.0f} layered {res[(n, 64)]:.0f}"
        for n in (1, 16, 64)), flush=True)
    assert res[(1, 64)] < res[(1, 0)]


@pytest.mark.parametrize("n,max_batch", [(6, 64), (100, 256)])
def test_queue_rows_that_are_not_binary_go_in_as_bytes(be, n, max_batch):
    """The queue packs the rows of small batches one bit per plane for the
    layered stem; a batch with a plane byte other than 0 / 1 goes in as
    bytes, so it still equals a direct forward of the same bytes, as does a
    batch too large for the layered kernels (a graph replay of bytes)."""
    import leela_amd
    from leela_amd.backend import DONE_FN
    p = leela_amd.PREC_FP16
    print(f"case: n={n} max_batch={max_batch}", flush=True)
    planes = make_batch(n, seed0=991)
    planes[2, 7, 100] = 2  # not a binary plane value
    be.set_layered_max(64)
    want_raw, want = be.forward(leela_amd.NET_POLICY, p, planes)
    got = np.full((n, 361), np.nan, np.float32)
    status = np.full(n, -99, np.int32)

    def done(user, st, raw, out):
        i = int(user or 0)
        status[i] = st
        if st == 0:
            got[i] = np.ctypeslib.as_array(out, (361,))
    cb = DONE_FN(done)
    be.queue_start(p, max_batch, 2000)
    try:
        for i in range(n):
            be.submit(leela_amd.NET_POLICY, planes[i], cb, i)
        be.join()
    finally:
        be.queue_stop()
    assert (status == 0).all()
    np.testing.assert_array_equal(got, want)
    # and the 2 matters: the same row with a 1 there differs
    planes[2, 7, 100] = 1
    _, other = be.forward(leela_amd.NET_POLICY, p, planes)
    assert not np.array_equal(other[2], want[2])
